"""Unit vectors and gated norms of heads in whole 16-byte pieces and in none, at the edges of what a lane holds."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# a piece, half a wave of them, a wave, two a lane, more than the kernels in pieces take; and parts that are no pieces
PARTS = [4, 12, 124, 128, 132, 256, 260, 512, 516, 7, 130]


@pytest.mark.parametrize("part", PARTS)
@pytest.mark.parametrize("heads, off", [(3, 0), (5, 4), (2, 3)])
def test_heads_as_unit_vectors(part, heads, off):
    g = torch.Generator().manual_seed(part)
    x = torch.randn(13, off + heads * part + 4 - off % 4, generator=g)
    got = ops.head_prepare(x.to(DEV), off, heads, part, unit=True, unit_eps=1e-6, n_first=1, scale_first=0.25, scale_rest=3.0).cpu()
    y = x[:, off:off + heads * part].double().view(13, heads, part)
    want = y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6) * torch.tensor([0.25] + [3.0] * (heads - 1))[:, None].double()
    # (a sum of `part` squares, a root, a division and two products of float32: under 2^-20 of a number in any order)
    torch.testing.assert_close(got[:, off:off + heads * part].double().view(13, heads, part), want, rtol=2 ** -20, atol=0)
    assert torch.equal(got[:, :off], x[:, :off]) and torch.equal(got[:, off + heads * part:], x[:, off + heads * part:])


@pytest.mark.parametrize("part", PARTS)
@pytest.mark.parametrize("gate_off", [0, 4, 1])
@pytest.mark.parametrize("gate_first, act, weighted", [(True, "silu", True), (False, "sigmoid", False)])
def test_gated_norms_of_parts(part, gate_off, gate_first, act, weighted):
    groups, n, eps = 3, 11, 1e-5
    g = torch.Generator().manual_seed(part + gate_off)
    x, gate = torch.randn(n, groups * part, generator=g), torch.randn(n, gate_off + groups * part + (-gate_off) % 4, generator=g)
    w = torch.randn(groups * part, generator=g)
    out = torch.empty(n, groups * part, device=DEV)
    ops.gated_group_norm(x.to(DEV), gate.to(DEV), gate_off, w.to(DEV) if weighted else None, groups, eps, out, gate_first, act)
    y, f = x.double(), gate[:, gate_off:gate_off + groups * part].double()
    f = torch.sigmoid(f) * (f if act == "silu" else 1.0)
    y = (y * f if gate_first else y).view(n, groups, part)
    y = (y * torch.rsqrt((y * y).mean(-1, keepdim=True) + eps)).view(n, -1) * (w.double() if weighted else 1.0)
    want = y if gate_first else y * f
    # (as above, and the gate's exponential and division)
    torch.testing.assert_close(out.cpu().double(), want, rtol=2 ** -19, atol=1e-30)
    half = torch.empty(n, groups * part, device=DEV, dtype=torch.bfloat16)
    ops.gated_group_norm(x.to(DEV), gate.to(DEV), gate_off, w.to(DEV) if weighted else None, groups, eps, half, gate_first, act)
    assert torch.equal(half, out.bfloat16())


@pytest.mark.parametrize("part", [4, 12, 60, 64, 68, 124, 128, 132, 192, 256])
@pytest.mark.parametrize("unit", [True, False])
def test_heads_in_pieces_have_the_general_kernels_bits(part, unit):
    """Rows that start one number further on, off every 16 bytes, go through the kernel for heads of any length."""
    n, heads = 700, 6
    x = torch.randn(n, heads * part + 8, generator=torch.Generator().manual_seed(part))
    x[0, 4:4 + part] *= 1e20                                  # (squares that overflow)
    x[1, 4] = float("inf")
    moved = torch.roll(x, 1, 1)
    got = [ops.head_prepare(rows.to(DEV), off, heads, part, unit=unit, unit_eps=1e-6, n_first=2, scale_first=0.3, scale_rest=1.7)
           .cpu()[:, off:off + heads * part] for rows, off in ((x, 4), (moved, 5))]
    assert torch.equal(*(t.view(torch.int32) for t in got)) or torch.equal(*(torch.nan_to_num(t, nan=7e7) for t in got))


@pytest.mark.parametrize("part, n", [(4, 600), (32, 600), (36, 600), (64, 600), (64, 1400), (68, 600), (96, 600), (96, 5500), (100, 5500), (128, 600),
                                     (100, 21900), (128, 21900), (132, 600), (256, 600), (260, 600), (388, 600), (512, 600)])
@pytest.mark.parametrize("gate_first, act, gated", [(True, "silu", True), (False, "sigmoid", True), (False, "silu", False)])
def test_gated_norms_in_pieces_have_the_general_kernels_bits(part, n, gate_first, act, gated):
    """Gates one number further on go through the kernel for parts of any length; without gates, rows that start off 16 bytes. Few and
    many parts, which take different kernels."""
    groups = 3
    g = torch.Generator().manual_seed(part)
    x, gate = torch.randn(n, groups * part, generator=g), torch.randn(n, groups * part + 8, generator=g)
    w = torch.randn(groups * part, generator=g).to(DEV)
    got = []
    for off in (4, 5):
        out = torch.empty(n, groups * part, device=DEV)
        flat = torch.empty(n * groups * part + off, device=DEV)[off:] if not gated else torch.empty(n * groups * part, device=DEV)
        rows = flat.view(n, groups * part).copy_(x)
        gates = torch.roll(gate, off - 4, 1).to(DEV) if gated else None
        ops.gated_group_norm(rows, gates, off if gated else 0, w, groups, 1e-5, out, gate_first, act)
        got.append(out.cpu())
    assert torch.equal(*got)

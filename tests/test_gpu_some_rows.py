"""Products of 17 to 128 rows at the edges of how they are shared out: tiles of rows, weight rows a block, chunks of K, slices."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 2.0 ** -24


def rnd(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


# one block partly past the end, a last block with one column or with four; one chunk of K, as many as are kept ahead, one more,
# nine; slices of unequal length (1,024 by 4,608 in eight)
SHAPES = [(8, 128), (41, 512), (100, 640), (1000, 1152), (3072, 256), (6148, 384), (1024, 4608)]


@pytest.mark.parametrize("n, k", SHAPES)
@pytest.mark.parametrize("m", [17, 32, 33, 48, 49, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("variant", [0, 616, 632, 664])
def test_some_rows_against_float64(m, n, k, variant):
    xg, wg, bg = (t.to(DEV) for t in (rnd(m, k, seed=1).bfloat16(), rnd(n, k, seed=2, scale=0.1).bfloat16(), rnd(n, seed=3)))
    plain = xg.double() @ wg.double().t() + bg.double()
    # a float32 sum of k products in any order: k roundings of at most the sum of their sizes
    bound = (xg.double().abs() @ wg.double().abs().t() + bg.double().abs()) * (k + 2) * EPS
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(xg, wg, out, bias=bg, variant=variant)
    assert bool(((out.double() - plain).abs() <= bound).all())
    half = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    ops.gemm(xg, wg, half, bias=bg, variant=variant)
    assert torch.equal(half, out.bfloat16())
    slices = ops.gemm_slices(m, n, k, torch.bfloat16)
    if slices > 1:
        parts = torch.full((slices, m, n), float("nan"), device=DEV)
        ops.gemm(xg, wg, parts, bias=bg, variant=variant)
        assert bool(((parts.double().sum(0) - plain).abs() <= bound).all())
    if not variant and ops.gemm_adds(m, n, k, torch.bfloat16):
        held = rnd(m, n, seed=4).to(DEV)
        added = held.clone()
        ops.gemm(xg, wg, added, bias=bg, add=True)
        torch.testing.assert_close(added, held + out, rtol=2e-6, atol=2e-5)     # (float32 results of unit size, one more rounding)
    if n % 2 == 0:
        g, u = out.double()[:, 0::2], out.double()[:, 1::2]
        for dtype, rtol in ((torch.float32, 4e-6), (torch.bfloat16, 5e-3)):
            gated = torch.empty(m, n // 2, device=DEV, dtype=dtype)
            ops.gemm(xg, wg, gated, bias=bg, swiglu=True, variant=variant)
            torch.testing.assert_close(gated.double(), g / (1.0 + torch.exp(-g)) * u, rtol=rtol, atol=1e-6)


def test_rows_that_start_anywhere_in_the_output():
    """Vectors go where the output is aligned for them, single values elsewhere."""
    x, w = rnd(40, 256, seed=5).bfloat16().to(DEV), rnd(64, 256, seed=6).bfloat16().to(DEV)
    want, got = torch.empty(40, 64, device=DEV, dtype=torch.bfloat16), torch.zeros(40 * 64 + 8, device=DEV, dtype=torch.bfloat16)
    ops.gemm(x, w, want)
    for at in (1, 2, 4):
        ops.gemm(x, w, got[at:at + 40 * 64].view(40, 64))
        assert torch.equal(got[at:at + 40 * 64].view(40, 64), want)
    gated = torch.empty(40, 32, device=DEV, dtype=torch.bfloat16)
    ops.gemm(x, w, gated, swiglu=True)
    ops.gemm(x, w, got[1:1 + 40 * 32].view(40, 32), swiglu=True)
    assert torch.equal(got[1:1 + 40 * 32].view(40, 32), gated)

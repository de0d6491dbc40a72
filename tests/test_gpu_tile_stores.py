"""How tiles of many rows leave: single values where a row's length or start does not allow pairs, on tiles that lie whole inside
the output and on cut ones."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 2.0 ** -24


def rnd(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def at(start, rows, columns, dtype):
    """[rows, columns] that starts `start` elements into a buffer, and the buffer."""
    buffer = torch.full((rows * columns + 16,), 7.0, device=DEV, dtype=dtype)
    return buffer[start:start + rows * columns].view(rows, columns), buffer


VARIANTS = [258, 263, 262, 358, 352, 558, 452, 351, 451]      # (four stages take K-steps in fours)


# several whole tiles and cut ones, rows of odd length and of even; 0: the plan's choice
@pytest.mark.parametrize("n", [1001, 1002])
@pytest.mark.parametrize("variant", VARIANTS + [0])
@pytest.mark.parametrize("start", [0, 1])
def test_single_values_and_pairs(n, variant, start):
    m, k = 700, 512
    x, w, b = (t.to(DEV) for t in (rnd(m, k, seed=1).bfloat16(), rnd(n, k, seed=2, scale=0.1).bfloat16(), rnd(n, seed=3)))
    plain = x.double() @ w.double().t() + b.double()
    # a float32 sum of k products in any order: k roundings of at most the sum of their sizes
    bound = (x.double().abs() @ w.double().abs().t() + b.double().abs()) * (k + 2) * EPS
    out, buffer = at(start, m, n, torch.float32)
    ops.gemm(x, w, out, bias=b, variant=variant)
    assert bool(((out.double() - plain).abs() <= bound).all())
    half, halves = at(start, m, n, torch.bfloat16)
    ops.gemm(x, w, half, bias=b, variant=variant)
    assert torch.equal(half, out.bfloat16())
    for kept, size in ((buffer, m * n), (halves, m * n)):
        assert bool((kept[:start] == 7).all()) and bool((kept[start + size:] == 7).all())
    if n % 2:
        return
    g, u = out.double()[:, 0::2], out.double()[:, 1::2]
    for dtype, rtol in ((torch.float32, 4e-6), (torch.bfloat16, 2.0 ** -8 + 1e-5)):
        gated, kept = at(start, m, n // 2, dtype)
        ops.gemm(x, w, gated, bias=b, swiglu=True, variant=variant)
        torch.testing.assert_close(gated.double(), g / (1.0 + torch.exp(-g)) * u, rtol=rtol, atol=1e-6)
        assert bool((kept[:start] == 7).all()) and bool((kept[start + m * n // 2:] == 7).all())


@pytest.mark.parametrize("n, start", [(1001, 0), (1001, 1), (1024, 1)])
def test_added_at_any_start(n, start):
    m, k = 700, 384
    assert ops.gemm_adds(m, n, k, torch.bfloat16) and ops.gemm_slices(m, n, k, torch.bfloat16) == 1
    x, w = rnd(m, k, seed=1).bfloat16().to(DEV), rnd(n, k, seed=2, scale=0.1).bfloat16().to(DEV)
    held, plain = rnd(m, n, seed=4).to(DEV), torch.empty(m, n, device=DEV)
    ops.gemm(x, w, plain)
    out, buffer = at(start, m, n, torch.float32)
    out.copy_(held)
    ops.gemm(x, w, out, add=True)
    assert torch.equal(out, held + plain)
    assert bool((buffer[:start] == 7).all()) and bool((buffer[start + m * n:] == 7).all())

"""Float32 products of more than 16 rows, on both tiles and at the edges of how K is walked, bit for bit."""
import numpy as np
import pytest
import torch

from imparo_amd.kernels import ops
from imparo_amd.kernels import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"

# less than a vector, a vector, around one step (32 or 64 of K), around the end of a turn of four and of the five behind it, and
# ends inside a vector
KS = [3, 4, 5, 31, 32, 33, 63, 64, 65, 66, 129, 160, 161, 194, 256, 257, 320, 322, 385, 513, 1026]


@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("m, n", [(17, 34), (70, 129), (400, 2050)])     # 32x32 twice, 64x64
@pytest.mark.parametrize("off", [0, 1])
def test_float32_tiles_sum_in_the_order_of_k(m, n, k, off):
    g = torch.Generator().manual_seed(k)
    x, w, b = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(n, generator=g)
    xg = torch.empty(m * k + off, device=DEV)[off:].view(m, k).copy_(x)      # (off 1: rows that start 4 bytes off 16)
    wg = torch.empty(n * k + off, device=DEV)[off:].view(n, k).copy_(w)
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(xg, wg, out)
    assert np.array_equal(out.cpu().numpy(), R.gemm(x, w))
    ops.gemm(xg, wg, out, bias=b.to(DEV))
    assert np.array_equal(out.cpu().numpy(), R.gemm(x, w, b))
    half = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    ops.gemm(xg, wg, half, bias=b.to(DEV))
    assert torch.equal(half, out.bfloat16())
    if n % 2 == 0:
        gated, gu = torch.empty(m, n // 2, device=DEV), R.gemm(x, w)
        ops.gemm(xg, wg, gated, swiglu=True)
        # (gate and up are the same bits: one exponential, one division and two products of float32 each)
        np.testing.assert_allclose(gated.cpu().numpy(), R.swiglu(gu[:, 0::2], gu[:, 1::2]), rtol=2e-6, atol=1e-6)



def test_float32_rows_do_not_depend_on_the_tile():
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(640, 520, generator=g).to(DEV), torch.randn(1024, 520, generator=g).to(DEV)
    whole = torch.empty(640, 1024, device=DEV)
    ops.gemm(x, w, whole)
    for m in (1, 16, 17, 64, 200, 333, 639):
        some = torch.empty(m, 1024, device=DEV)
        ops.gemm(x[:m], w, some)
        assert torch.equal(some, whole[:m])

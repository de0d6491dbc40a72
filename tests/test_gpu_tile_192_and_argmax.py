"""The 192-row tile at the edges of its tiles, and argmax where its two passes meet special rows."""
import math

import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 2.0 ** -24


@pytest.mark.parametrize("m", [65, 192, 193, 384, 520])
@pytest.mark.parametrize("n, k", [(256, 128), (250, 256), (514, 1152)])
def test_tile_of_192_rows_against_float64(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).bfloat16().to(DEV), (torch.randn(n, k, generator=g) * 0.1).bfloat16().to(DEV)
    b = torch.randn(n, generator=g).to(DEV)
    plain = x.double() @ w.double().t() + b.double()
    bound = (x.double().abs() @ w.double().abs().t() + b.double().abs()) * (k + 2) * EPS
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(x, w, out, bias=b, variant=558)
    assert bool(((out.double() - plain).abs() <= bound).all())
    gated = torch.full((m, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm(x, w, gated, bias=b, swiglu=True, variant=558)
    u, v = out.double()[:, 0::2], out.double()[:, 1::2]
    torch.testing.assert_close(gated.double(), u / (1.0 + torch.exp(-u)) * v, rtol=2.0 ** -8 + 1e-5, atol=1e-6)


@pytest.mark.parametrize("m, n, k", [(151, 69516, 3584), (167, 67434, 3584)])
def test_the_tile_takes_no_slices_place(m, n, k):
    """Two slices of K are nearer to 64 bits than one piece: these shapes had two before there was the tile."""
    assert ops.gemm_slices(m, n, k, torch.bfloat16) == 2


@pytest.mark.parametrize("vocab", [64, 4096, 65536, 65540, 200000])
def test_argmax_of_special_rows(vocab):
    g = torch.Generator().manual_seed(vocab)
    rows = torch.randn(9, vocab, generator=g)
    rows[1] = -math.inf                                         # the first index
    rows[2] = math.nan
    rows[3], rows[3, vocab - 1] = -math.inf, -1e30              # one number among -inf, in the last piece
    rows[4] = 7.0                                               # all equal: the first index
    rows[5, [vocab // 2, vocab - 1, vocab // 2 + 1]] = 50.0     # ties across threads and runs of loads
    rows[6], rows[6, 5] = math.nan, -math.inf                   # -inf among NaN
    rows[7, 3], rows[7, vocab - 2] = math.nan, math.inf
    want = [int(rows[0].argmax()), 0, 0, vocab - 1, 0, vocab // 2, 5, vocab - 2, int(rows[8].argmax())]
    out = torch.empty(9, device=DEV, dtype=torch.int32)
    ops.argmax_rows(rows.to(DEV), out)
    assert out.tolist() == want

"""Products of at most 16 rows at the edges of how they are shared out: tiles a block, chunks of K a wave, rounds, ragged K."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 2.0 ** -24


def rnd(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


# (n, k): one tile and a part of one, two, three and four tiles a block (256, 512, 768 tiles and beyond), a last block whose
# tiles are partly or wholly past the end; one chunk of K, nine (three a wave), ten, 17, 32 and 33 (a second round); a K
# that is no multiple of 128, and shorter than a lane's part of a chunk
SHAPES = [(16, 128), (4, 8), (41, 72), (130, 1152), (4096, 256), (4100, 1280), (8200, 640), (12296, 128), (16360, 256), (17000, 136),
          (70, 2176), (33, 4096), (18, 4224), (258, 5128), (4112, 2112)]


@pytest.mark.parametrize("n, k", SHAPES)
@pytest.mark.parametrize("m", [1, 5, 16])
def test_few_rows_against_float64(m, n, k):
    x, w, b = rnd(m, k, seed=1).bfloat16(), rnd(n, k, seed=2, scale=0.1).bfloat16(), rnd(n, seed=3)
    xg, wg, bg = x.to(DEV), w.to(DEV), b.to(DEV)
    plain = (xg.double() @ wg.double().t() + bg.double()).cpu()
    # a float32 sum of k products in any order: k roundings of at most the sum of their sizes
    bound = (xg.double().abs() @ wg.double().abs().t() + bg.double().abs()).cpu() * (k + 2) * EPS
    out = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(xg, wg, out, bias=bg)
    assert bool(((out.cpu().double() - plain).abs() <= bound).all())
    half = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    ops.gemm(xg, wg, half, bias=bg)
    assert torch.equal(half.cpu(), out.cpu().bfloat16())
    slices = ops.gemm_slices(m, n, k, torch.bfloat16)
    if slices > 1:
        parts = torch.full((slices, m, n), float("nan"), device=DEV)
        ops.gemm(xg, wg, parts, bias=bg)
        assert bool(((parts.double().sum(0).cpu() - plain).abs() <= bound).all())
    # every row by itself gives the bits it has among others, whatever the tiles a block that the row count chooses
    for r in {0, m - 1}:
        one = torch.empty(1, n, device=DEV)
        ops.gemm(xg[r:r + 1].contiguous(), wg, one, bias=bg)
        assert torch.equal(one[0], out[r])
    if n % 2 == 0:
        gated = torch.empty(m, n // 2, device=DEV)
        ops.gemm(xg, wg, gated, bias=bg, swiglu=True)
        g, u = out.cpu().double()[:, 0::2], out.cpu().double()[:, 1::2]
        torch.testing.assert_close(gated.cpu().double(), g / (1.0 + torch.exp(-g)) * u, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("parts", [1, 31, 128, 256, 600])
@pytest.mark.parametrize("m, k", [(1, 128), (3, 1024), (16, 2176)])
def test_rows_scaled_at_the_end(m, k, parts):
    """The partial sums of squares of fewer parts than threads, of a whole round of loads and of more than one."""
    x, w = rnd(m, k, seed=5).bfloat16().to(DEV), rnd(96, k, seed=6, scale=0.1).bfloat16().to(DEV)
    ssq = torch.zeros(parts, 16)
    ssq[:, :m] = rnd(parts, m, seed=7).square() + 0.1
    out, plain = torch.empty(m, 96, device=DEV), torch.empty(m, 96, device=DEV)
    ops.rows_gemm(x, w, out=out, ssq_in=ssq.to(DEV), eps=1e-5)
    ops.rows_gemm(x, w, out=plain)
    scale = torch.rsqrt(ssq.double()[:, :m].sum(0) / k + 1e-5)
    torch.testing.assert_close(out.cpu().double(), plain.cpu().double() * scale[:, None], rtol=parts * EPS + 1e-6, atol=0.0)

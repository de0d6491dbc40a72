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


@pytest.mark.parametrize("n, k", [(1000, 1152), (520, 2048), (1024, 4608)])
@pytest.mark.parametrize("m", [17, 64, 65, 128])
@pytest.mark.parametrize("variant", [0, 616, 632, 664])
def test_walks_longer_than_the_chunks_kept_ahead_add_in_float32(m, n, k, variant):
    """The bound above grows with K until sums kept in 16 bits would pass it: a row's relative error over all columns instead. A
    quarter's sum takes k / 128 products of 32 k, each added with two roundings at most of up to 2^-24 of a partial sum; these are
    independent, and of partial sums that grow as the root of how many products they hold: sqrt(k / 128) 2^-24 in all, and three
    more roundings where the quarters meet."""
    most = (k / 128 + 3) ** 0.5 * EPS
    x, w = rnd(m, k, seed=1).bfloat16().to(DEV), rnd(n, k, seed=2, scale=0.1).bfloat16().to(DEV)
    plain, out = x.double() @ w.double().t(), torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(x, w, out, variant=variant)
    assert float(((out.double() - plain).norm(dim=1) / plain.norm(dim=1)).max()) <= most
    slices = ops.gemm_slices(m, n, k, torch.bfloat16)
    if slices > 1:
        parts = torch.full((slices, m, n), float("nan"), device=DEV)
        ops.gemm(x, w, parts, variant=variant)
        assert float(((parts.double().sum(0) - plain).norm(dim=1) / plain.norm(dim=1)).max()) <= most


# a K that is no multiple of 128 (the kernel that shares staged activations between waves, and behind it tiles staged through
# registers), and the numbers of rows around where tiles of 128 rows take over from this file's kernel with wide weights
@pytest.mark.parametrize("m, n, k", [(24, 12362, 1032), (64, 12362, 1032), (40, 1000, 1032), (65, 1000, 1032), (96, 16384, 512), (97, 16384, 512),
                                     (128, 16384, 512), (97, 16384, 1536), (97, 1024, 512), (129, 1024, 512)])
def test_where_other_kernels_begin(m, n, k):
    x, w, b = (t.to(DEV) for t in (rnd(m, k, seed=1).bfloat16(), rnd(n, k, seed=2, scale=0.1).bfloat16(), rnd(n, seed=3)))
    plain, out = x.double() @ w.double().t() + b.double(), torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(x, w, out, bias=b)
    # (as above, but a column's sum is one chain of k / 16 products: sqrt(k / 16) 2^-24)
    assert float(((out.double() - plain).norm(dim=1) / plain.norm(dim=1)).max()) <= (k / 16 + 3) ** 0.5 * EPS
    half = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    ops.gemm(x, w, half, bias=b)
    assert torch.equal(half, out.bfloat16())
    g, u = out.double()[:, 0::2], out.double()[:, 1::2]
    gated = torch.empty(m, n // 2, device=DEV)
    ops.gemm(x, w, gated, bias=b, swiglu=True)
    torch.testing.assert_close(gated.double(), g / (1.0 + torch.exp(-g)) * u, rtol=4e-6, atol=1e-6)


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

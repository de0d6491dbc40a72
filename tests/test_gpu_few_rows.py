"""Products of at most 16 rows at the edges of how they are shared out: tiles a block, chunks of K a wave, rounds, ragged K."""
import math

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


# K of less than a run, ragged, one round of runs and more than one; experts that nobody chose, so that the list ends in
# empty tiles (many tiles, and a last tile of weight rows partly past the end: below)
@pytest.mark.parametrize("n, k", [(64, 8), (192, 72), (1536, 1024), (1088, 136), (64, 2120), (832, 768)])
@pytest.mark.parametrize("tokens, experts, top", [(1, 3, 2), (8, 9, 4), (16, 4, 4)])
def test_experts_products_of_few_rows(n, k, tokens, experts, top):
    g = torch.Generator().manual_seed(n + k + tokens)
    choice = torch.stack([torch.randperm(max(top, experts - 2), generator=g)[:top] for _ in range(tokens)]).int()
    entries = tokens * top
    rows = ops.moe_tile_rows(entries, experts, torch.bfloat16)
    assert rows == 16
    tiles = torch.empty(ops.moe_max_tiles(entries, experts, rows), 3, device=DEV, dtype=torch.int32)
    slot, entry = torch.empty(entries, device=DEV, dtype=torch.int32), torch.empty(entries, device=DEV, dtype=torch.int32)
    ops.moe_plan(choice.to(DEV), experts, rows, slot, entry, tiles)
    x, w = rnd(tokens, k, seed=1).bfloat16().to(DEV), rnd(experts, n, k, seed=2, scale=0.1).bfloat16().to(DEV)
    weight = torch.rand(entries, generator=g).to(DEV)
    per_entry, expert = x.double().repeat_interleave(top, 0), choice.flatten().long().to(DEV)
    plain = torch.bmm(w.double()[expert], per_entry[:, :, None])[:, :, 0]
    bound = torch.bmm(w.double().abs()[expert], per_entry.abs()[:, :, None])[:, :, 0] * (k + 2) * EPS
    at = slot.long()
    out = torch.full((entries, n), float("nan"), device=DEV)
    ops.moe_gemm(x, w, out, tiles, rows, entry_of_slot=entry, gather_div=top)
    assert bool(((out[at].double() - plain).abs() <= bound).all())
    half = torch.empty(entries, n, device=DEV, dtype=torch.bfloat16)
    ops.moe_gemm(x, w, half, tiles, rows, entry_of_slot=entry, gather_div=top)
    assert torch.equal(half, out.bfloat16())
    gated = torch.full((entries, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.moe_gemm(x, w, gated, tiles, rows, entry_of_slot=entry, gather_div=top, epilogue="gated", weight=weight)
    z = out[at].double().view(entries, n // 64, 2, 32) * weight.double()[:, None, None, None]
    want = (z[:, :, 0] / (1.0 + torch.exp(-z[:, :, 0])) * z[:, :, 1]).reshape(entries, n // 2)
    torch.testing.assert_close(gated[at].double(), want, rtol=2.0 ** -8 + 1e-5, atol=1e-6)


# float32 through the ring: fewer chunks of 64 than stages, as many, an odd number, more than one turn; weight rows that are no
# multiple of 16; one load of activations a stage and four; a K that goes the other way; few blocks and more than 512
@pytest.mark.parametrize("n, k", [(5, 64), (33, 256), (70, 704), (40, 768), (16, 832), (130, 1600), (8200, 320), (24, 68)])
@pytest.mark.parametrize("m", [1, 4, 5, 16])
def test_float32_few_rows_are_the_many_rows_bits(m, n, k):
    x, w, b = rnd(20, k, seed=1).to(DEV), rnd(n, k, seed=2, scale=0.1).to(DEV), rnd(n, seed=3).to(DEV)
    many = torch.empty(20, n, device=DEV)
    ops.gemm(x, w, many, bias=b)                 # (more than 16 rows: the tile kernel, held to the statement elsewhere)
    few = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm(x[:m].contiguous(), w, few, bias=b)
    assert torch.equal(few, many[:m])
    if n % 2 == 0:
        many, few = torch.empty(20, n // 2, device=DEV), torch.full((m, n // 2), float("nan"), device=DEV)
        ops.gemm(x, w, many, bias=b, swiglu=True)
        ops.gemm(x[:m].contiguous(), w, few, bias=b, swiglu=True)
        assert torch.equal(few, many[:m])


# K that is no multiple of 128: the last eight activations are what a chunk would read again past K
@pytest.mark.parametrize("k", [8, 24, 136, 392, 1032, 1288, 2312, 5000])
def test_an_infinite_last_activation_stays_one(k):
    m, n = 3, 48
    x, w = rnd(m, k, seed=1).bfloat16(), rnd(n, k, seed=2, scale=0.1).bfloat16()
    x[1, k - 1] = math.inf
    want = (w[:, k - 1].float().sign() * math.inf).to(DEV)
    finite = x.clone()
    finite[1, k - 1] = 0.0
    xg, fg, wg = x.to(DEV), finite.to(DEV), w.to(DEV)
    out, plain, rows = (torch.empty(m, n, device=DEV) for _ in range(3))
    ops.gemm(fg, wg, plain)
    ops.gemm(xg, wg, out)
    ops.rows_gemm(xg, wg, out=rows)
    stream, ssq = torch.zeros(m, n, device=DEV), torch.empty(ops.rows_parts(n), 16, device=DEV)
    ops.rows_gemm(xg, wg, into=stream, ssq_out=ssq)
    for y in (out, rows, stream):
        assert torch.equal(y[1], want)
        assert torch.equal(y[[0, 2]], plain[[0, 2]]) or y is stream
    # the conv's input projection: B, C and x of the row are infinite, one tap of 1 on the token itself
    e = n // 3
    state, slot = torch.zeros(m, 1, e, device=DEV), torch.arange(m, device=DEV, dtype=torch.int32)
    conv, taps = torch.empty(m, e, device=DEV), torch.tensor([[0.0, 1.0]] * e, device=DEV)
    ops.in_proj_conv_decode(xg, wg, None, taps, None, state, slot, conv)
    b, c, u = want[:e], want[e:2 * e], want[2 * e:]
    assert torch.equal(conv[1], c * (b * u)) and bool(conv[[0, 2]].isfinite().all())


# The root mean square of the errors against 64 bits, in units of the outputs', goes by how many chains of sums a column has
# and how long they are: eight chains of two chunks of 128 at the most up to K = 2,048 and sixteen beyond measured 8.8e-8,
# 9.8e-8, 1.02e-7, 1.04e-7, 1.09e-7 and 1.15e-7 here; three to seven waves with longer chains 1.15e-7, 9.9e-8, 1.2e-7, 1.2e-7,
# 1.2e-7 and 1.35e-7. The limits lie between (16,384 outputs of independent roundings: the figures stray by less than 1 %).
@pytest.mark.parametrize("k, limit", [(1152, 1.0e-7), (1920, 1.1e-7), (2304, 1.1e-7), (2560, 1.12e-7), (3584, 1.24e-7)])
def test_sums_stay_as_near_to_64_bits(k, limit):
    m, n = 16, 1024
    x, w = rnd(m, k, seed=1).bfloat16().to(DEV), rnd(n, k, seed=2, scale=0.02).bfloat16().to(DEV)
    out = torch.empty(m, n, device=DEV)
    ops.rows_gemm(x, w, out=out)
    want = x.double() @ w.double().t()
    assert float((out.double() - want).norm() / want.norm()) < limit


# every way to share a product out: three and four tiles a block with one, two and three chunks in flight, walks of several
# rounds with waves that have a chunk less, turned walks whose rounds end unevenly, pairs of chunks, slices of two rounds
@pytest.mark.parametrize("n, k", [(9200, 1152), (9216, 3072), (12288, 2304), (17600, 3072), (20010, 2312), (24576, 2048), (6144, 5504),
                                  (9000, 4224), (12300, 4608), (16400, 6144), (3072, 12288), (2048, 16384), (1030, 14336), (70, 8968)])
def test_few_rows_have_the_same_bits_however_they_are_shared_out(n, k):
    x, w = rnd(16, k, seed=1).bfloat16().to(DEV), rnd(n, k, seed=2, scale=0.02).bfloat16().to(DEV)
    plain, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    whole = torch.full((16, n), float("nan"), device=DEV)
    ops.rows_gemm(x, w, out=whole)
    assert bool(((whole.double() - plain).abs() <= size * (k + 2) * EPS).all())
    ssq = torch.full((1, 16), float(k), device=DEV)          # (a scale of one, but for eps)
    for m in (1, 2, 4, 5, 9):
        out = torch.full((m, n), float("nan"), device=DEV)
        ops.rows_gemm(x[:m].contiguous(), w, out=out)
        assert torch.equal(out, whole[:m])
        ops.rows_gemm(x[:m].contiguous(), w, out=out, ssq_in=ssq, eps=1e-12)
        assert torch.equal(out, whole[:m])
    slices = ops.gemm_slices(16, n, k, torch.bfloat16)
    if slices > 1:
        parts, one = torch.full((slices, 16, n), float("nan"), device=DEV), torch.full((slices, 1, n), float("nan"), device=DEV)
        ops.gemm(x, w, parts)
        ops.gemm(x[3:4].contiguous(), w, one)
        assert bool(((parts.double().sum(0) - plain).abs() <= size * (k + 2) * EPS).all()) and torch.equal(one[:, 0], parts[:, 3])
    if n <= 9216:
        stream = torch.zeros(16, n, device=DEV)
        ssq = torch.full((ops.rows_parts(n), 16), float("nan"), device=DEV)
        ops.rows_gemm(x, w, into=stream, ssq_out=ssq)
        assert bool(((stream.double() - plain).abs() <= size * (k + 2) * EPS).all())
        torch.testing.assert_close(ssq.double().sum(0), stream.double().square().sum(1), rtol=1e-5, atol=0.0)


# more tiles of weight rows than blocks run at once, a last one partly past the end, waves without a run (K up to 128), with one
# to five; lists with an empty tile at the end and without one, and lists that do not count them
@pytest.mark.parametrize("n, k", [(1700, 136), (4100, 72), (1536, 1024), (1000, 320), (24, 8), (2050, 1288)])
@pytest.mark.parametrize("tokens, experts, top", [(8, 9, 5), (16, 40, 5), (1, 1, 1)])
def test_experts_products_of_many_tiles(n, k, tokens, experts, top):
    g = torch.Generator().manual_seed(n + k + tokens)
    choice = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(tokens)]).int()
    entries = tokens * top
    rows = ops.moe_tile_rows(entries, experts, torch.bfloat16)
    assert rows == 16
    tiles = torch.empty(ops.moe_max_tiles(entries, experts, rows), 3, device=DEV, dtype=torch.int32)
    slot, entry = torch.empty(entries, device=DEV, dtype=torch.int32), torch.empty(entries, device=DEV, dtype=torch.int32)
    ops.moe_plan(choice.to(DEV), experts, rows, slot, entry, tiles)
    x, w = rnd(tokens, k, seed=1).bfloat16().to(DEV), rnd(experts, n, k, seed=2, scale=0.1).bfloat16().to(DEV)
    expert, token = choice.flatten().long().to(DEV), torch.arange(entries, device=DEV) // top
    plain, size = (torch.empty(entries, n, device=DEV, dtype=torch.float64) for _ in range(2))
    for e in range(experts):
        of = expert == e
        plain[of] = x[token[of]].double() @ w[e].double().t()
        size[of] = x[token[of]].double().abs() @ w[e].double().abs().t()
    at = slot.long()
    out = torch.full((entries, n), float("nan"), device=DEV)
    ops.moe_gemm(x, w, out, tiles, rows, entry_of_slot=entry, gather_div=top)
    assert bool(((out[at].double() - plain).abs() <= size * (k + 2) * EPS).all())
    live = tiles[tiles[:, 0] >= 0]
    for listed in (live, torch.cat([live, torch.tensor([[-1, 0, 0]] * 3, device=DEV, dtype=torch.int32), live[:1]])):
        again = torch.full_like(out, float("nan"))
        ops.moe_gemm(x, w, again, listed.contiguous(), rows, entry_of_slot=entry, gather_div=top)
        assert torch.equal(again, out)
    if n % 64 == 0:
        gated = torch.full((entries, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.moe_gemm(x, w, gated, tiles, rows, entry_of_slot=entry, gather_div=top, epilogue="gated")
        z = out[at].double().view(entries, n // 64, 2, 32)
        want = (z[:, :, 0] / (1.0 + torch.exp(-z[:, :, 0])) * z[:, :, 1]).reshape(entries, n // 2)
        torch.testing.assert_close(gated[at].double(), want, rtol=2.0 ** -8 + 1e-5, atol=1e-6)

"""Float32 attention of few tokens: chunks of keys side by side over a block's waves, the bits of one wave's walk."""
import pytest
import torch

from gpu_helpers import hand_context

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def ops():
    from imparo_amd.kernels import ops
    return ops


@pytest.mark.parametrize("H,Hk,D", [(16, 8, 64), (4, 4, 64), (8, 2, 64), (6, 2, 128), (4, 1, 128), (5, 1, 64)])
@pytest.mark.parametrize("window,keep,capped", [(None, 0, False), (600, 70, True), (64, 0, False), (1, 130, True), (-100, 0, False)])
def test_few_tokens_have_the_general_kernels_bits(H, Hk, D, window, keep, capped):
    """Contexts at whole chunks and rounds of them (256 and 512 keys), beside them, and of one key; values transposed in their
    pages go through the general kernel."""
    lens, page = (1, 64, 65, 256, 257, 511, 513, 1100), 16
    R, n_pages = len(lens), sum(-(-c // page) for c in lens) + 2
    ctx = hand_context([(c - 1, 1) for c in lens], page, n_pages, torch.float32, DEV, kv_sites={0: (Hk, D)})
    table = ctx.block_tables[0]
    g = torch.Generator().manual_seed(1)
    k, v, q = (torch.randn(*s, generator=g).to(DEV) for s in ((n_pages, Hk, page, D), (n_pages, Hk, page, D), (R, H, D)))
    rule = None
    if keep or capped:
        rule = ops().attention_rule(H, keep_first=keep, softcap=8.0 if capped else None, sink=torch.randn(H, generator=g).to(DEV), out_scale=0.9)
    got = []
    for transposed in (False, True):
        out = torch.full((R, H * D), float("nan"), device=DEV)
        values = v.transpose(2, 3).contiguous() if transposed else v
        ops().attention(q, k, values, out, ctx.positions, ctx.row_of_token, table, 0.125, window, v_transposed=transposed, rule=rule)
        got.append(out.cpu())
    assert bool(torch.isfinite(got[0]).all()) and torch.equal(*got)


def test_pages_behind_two_billion_numbers():
    """A pool of more than 2^31 numbers (8 GiB of keys), keys in its last pages: a key's place is past what a signed int holds."""
    H, Hk, D, page, n = 4, 2, 64, 16, 70
    n_pages = 2 ** 31 // (Hk * page * D) + 40
    held = list(range(n_pages - 5, n_pages))
    ctx = hand_context([(n - 1, 1)], page, 8, torch.float32, DEV, kv_sites={0: (Hk, D)}, tables=[held])
    g = torch.Generator().manual_seed(2)
    k, v = (torch.empty(n_pages, Hk, page, D, device=DEV) for _ in range(2))
    q = torch.randn(1, H, D, generator=g)
    for cache in (k, v):
        cache[held] = torch.randn(len(held), Hk, page, D, generator=g).to(DEV)
    out = torch.full((1, H * D), float("nan"), device=DEV)
    wide = torch.full((1, 8), -1, dtype=torch.int32, device=DEV)         # (room for more than one chunk of 64 keys)
    wide[:, :len(held)] = ctx.block_tables[0]
    ops().attention(q.to(DEV), k, v, out, ctx.positions, ctx.row_of_token, wide, 0.125, None)
    keys, values = (c[held].cpu().double().transpose(0, 1).reshape(Hk, -1, D)[:, :n].repeat_interleave(H // Hk, 0) for c in (k, v))
    weights = torch.softmax((keys @ q[0].double()[:, :, None])[..., 0] * 0.125, -1)
    want = (weights[:, None] @ values)[:, 0].reshape(1, -1)
    # (sums of 64 and of 70 products in float32)
    torch.testing.assert_close(out.cpu().double(), want, rtol=2 ** -18, atol=2 ** -20)


@pytest.mark.parametrize("H,Hk,D", [(16, 8, 64), (32, 8, 64), (8, 2, 128)])
@pytest.mark.parametrize("page", [8, 32, 64])
@pytest.mark.parametrize("gated", [False, True])
def test_portions_gates_and_other_pages_have_the_general_kernels_bits(H, Hk, D, page, gated):
    """Several tokens of a request beside single ones, rows with a gate a head, pages of other sizes, rows of one chunk among long
    ones."""
    segments = [(0, 3), (60, 6), (63, 1), (300, 4), (40, 1), (700, 2)]
    T, n_pages = sum(n for _, n in segments), sum(-(-(p + n) // page) for p, n in segments) + 1
    ctx = hand_context(segments, page, n_pages, torch.float32, DEV, kv_sites={0: (Hk, D)})
    g = torch.Generator().manual_seed(page)
    k, v, q = (torch.randn(*s, generator=g).to(DEV) for s in ((n_pages, Hk, page, D), (n_pages, Hk, page, D), (T, H, D)))
    rule = ops().attention_rule(H, softcap=8.0, out_scale=0.9)
    if gated:
        rule = rule.with_gate(torch.randn(T, H + 4, generator=g).to(DEV), 4)
    got = []
    for transposed in (False, True):
        out = torch.full((T, H * D), float("nan"), device=DEV)
        ops().attention(q, k, v.transpose(2, 3).contiguous() if transposed else v, out, ctx.positions, ctx.row_of_token, ctx.block_tables[0],
                        0.125, None, v_transposed=transposed, rule=rule)
        got.append(out.cpu())
    assert bool(torch.isfinite(got[0]).all()) and torch.equal(*got)


@pytest.mark.parametrize("H,Hk,D", [(16, 8, 64), (32, 8, 64), (4, 1, 128), (2, 2, 128)])
@pytest.mark.parametrize("window", [None, 1, 16, 17, -64, -96])
def test_sixteens_of_a_walks_only_chunk_have_the_general_kernels_bits(H, Hk, D, window):
    """Contexts, and windows inside one run of 64 keys, that end or start on sixteens of its rows and beside them."""
    lens, page = (1, 15, 16, 17, 31, 33, 48, 49, 63, 64, 80, 97, 128), 16
    R, n_pages = len(lens), sum(-(-c // page) for c in lens) + 2
    ctx = hand_context([(c - 1, 1) for c in lens], page, n_pages, torch.float32, DEV, kv_sites={0: (Hk, D)})
    g = torch.Generator().manual_seed(2)
    k, v, q = (torch.randn(*s, generator=g).to(DEV) for s in ((n_pages, Hk, page, D), (n_pages, Hk, page, D), (R, H, D)))
    got = []
    for values, transposed in ((v, False), (v.transpose(2, 3).contiguous(), True)):
        out = torch.full((R, H * D), float("nan"), device=DEV)
        ops().attention(q, k, values, out, ctx.positions, ctx.row_of_token, ctx.block_tables[0], 0.125, window, v_transposed=transposed)
        got.append(out.cpu())
    assert bool(torch.isfinite(got[0]).all()) and torch.equal(*got)

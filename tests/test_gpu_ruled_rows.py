"""Decode attention under a rule out of the projection's rows: one launch instead of two."""
import math

import pytest
import torch

from gpu_helpers import hand_context

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def ops():
    from imparo_amd.kernels import ops
    return ops


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("over", ["head", "projection"])
@pytest.mark.parametrize("H,Hk,D", [(8, 2, 64), (20, 1, 64), (32, 16, 64)])
@pytest.mark.parametrize("window,keep,page", [(None, 0, 64), (300, 70, 64), (32, 33, 32), (1, 0, 16), (-100, 0, 64)])
@pytest.mark.parametrize("brings,gated,magnitude", [(True, False, 1.0), (True, True, 1.2), (False, False, 1.2)])
def test_ruled_attention_from_the_projection_rows(over, H, Hk, D, window, keep, page, brings, gated, magnitude):
    """Rows that bring queries, keys and values, or queries alone (another layer's cache), as the launch that norms, turns
    and stores and the launch that attends give them: bit for bit, but for norms a head, whose squares are added in another
    order and may turn a rounding to bfloat16. The row's own key is the first, the last of a tile, of a split, the first of one."""
    lens = (1, 32, 33, 256, 257, 512, 513, 700)
    R, n_pages = len(lens), sum(-(-c // page) for c in lens) + 2
    ctx = hand_context([(c - 1, 1) for c in lens], page, n_pages, torch.bfloat16, DEV, kv_sites={0: (Hk, D)}, v_transposed=True)
    k0, v0, table = ctx.kv(0)
    k0.copy_(rnd(*k0.shape, seed=1)), v0.copy_(rnd(*v0.shape, seed=2))
    units = H + (2 * Hk if brings else 0)
    width = units * D + ((H + 7) // 8 * 8 if gated else 0)
    rows = rnd(R, width, seed=3).to(DEV)
    whole = over == "projection"
    assert ops().attention_decode_qkv_ruled_takes(H, Hk, D, D // 2, whole)
    qw, kw = (1 + 0.1 * rnd(H * D if whole else D, seed=4)).to(DEV), (1 + 0.1 * rnd(Hk * D if whole else D, seed=5)).to(DEV)
    freq = torch.linspace(1.0, 0.01, D // 2, device=DEV)
    rule = ops().attention_rule(H, keep_first=keep, softcap=20.0, sink=rnd(H, seed=7).to(DEV), out_scale=0.7)
    if gated:
        rule = rule.with_gate(rows, units * D)
    scale = 1.0 / math.sqrt(D)
    seen = ops().attention_ruled_keys(max(lens), window, rule)
    splits = -(-seen // 256)
    part = lambda n: torch.full((R * H * splits * n,), float("nan"), device=DEV)
    got = []
    for one in (True, False):
        k, v = k0.clone(), v0.clone()
        out = torch.full((R, H * D), float("nan"), dtype=torch.bfloat16, device=DEV)
        tail = (part(D), part(2), ctx.single_rows, R, ctx.seg_start, ctx.positions, table)
        if one:
            ops().attention_decode_qkv(rows, qw, kw, 1e-5, freq, k, v, out, *tail, H, scale, window, max(lens), write_kv=brings,
                                       rule=rule, magnitude=magnitude, whole=whole)
        else:
            q = torch.empty(R, H, D, dtype=torch.bfloat16, device=DEV)
            ops().qk_row_norm_rope_store(rows, qw, kw, over, 1e-5, freq, magnitude, ctx.positions, ctx.row_of_token,
                                         table if brings else None, page, q, k if brings else None, v if brings else None, H,
                                         Hk if brings else 0, D, D, v_transposed=True)
            ops().attention_decode(q, k, v, out, *tail, scale, window, max(lens), exact=True, rule=rule)
        got.append((out.cpu().float(), k.cpu(), v.cpu()))
    assert bool(torch.isfinite(got[1][0]).all())
    if whole:
        assert all(torch.equal(a, b) for a, b in zip(*got))
    top = float(got[1][0].abs().max())
    torch.testing.assert_close(got[0][0], got[1][0], rtol=2 ** -6, atol=top * 2 ** -8)
    torch.testing.assert_close(got[0][1].float(), got[1][1].float(), rtol=2 ** -7, atol=2 ** -9)
    assert torch.equal(got[0][2], got[1][2])


def test_ruled_rows_of_a_wrong_width_are_refused():
    from imparo_amd.kernels import KernelArgumentError
    ctx = hand_context([(4, 1)], 64, 4, torch.bfloat16, DEV, kv_sites={0: (2, 64)}, v_transposed=True)
    k, v, table = ctx.kv(0)
    i = torch.zeros(1, dtype=torch.int32, device=DEV)
    out, part = torch.zeros(1, 4 * 64, dtype=torch.bfloat16, device=DEV), torch.zeros(4096, device=DEV)
    rule = ops().attention_rule(4, softcap=20.0)
    for width in (4 * 64, 8 * 64 + 2):
        with pytest.raises(KernelArgumentError):
            ops().attention_decode_qkv(torch.zeros(1, width, device=DEV), None, None, 0.0, None, k, v, out, part, part, i, 1, i, i,
                                       table, 4, 0.125, None, 5, rule=rule)
    takes = ops().attention_decode_qkv_ruled_takes
    assert takes(33, 33, 64, 32, False) and takes(8, 2, 64, 0, False) and not takes(8, 2, 64, 16, False)
    assert not takes(33, 1, 64, 32, True) and not takes(17, 17, 64, 32, True) and not takes(8, 2, 128, 64, False)


def _one_and_two_launches(rows, H, Hk, qw, kw, freq, over, lens, brings=True, magnitude=1.0, gated=False, interleaved=False, page=64):
    """(outputs, keys, values) of the one launch and of the two that it stands for, on the CPU."""
    R, D = rows.shape[0], 64
    ctx = hand_context([(c - 1, 1) for c in lens], page, sum(-(-c // page) for c in lens) + 2, torch.bfloat16, DEV,
                       kv_sites={0: (Hk, D)}, v_transposed=True)
    k0, v0, table = ctx.kv(0)
    k0.copy_(rnd(*k0.shape, seed=1)), v0.copy_(rnd(*v0.shape, seed=2))
    rule = ops().attention_rule(H, softcap=20.0, sink=rnd(H, seed=7).to(DEV))
    if gated:
        rule = rule.with_gate(rows, (H + 2 * Hk) * D)
    row_store = gated or over == "projection" or magnitude != 1.0           # (as the attention part chooses)
    more = dict(row_store=True) if row_store and over == "head" else {}
    splits = -(-ops().attention_ruled_keys(max(lens), None, rule) // 256)
    part = lambda n: torch.full((R * H * splits * n,), float("nan"), device=DEV)
    got = []
    for one in (True, False):
        k, v = k0.clone(), v0.clone()
        out = torch.full((R, H * D), float("nan"), dtype=torch.bfloat16, device=DEV)
        tail = (part(D), part(2), ctx.single_rows, R, ctx.seg_start, ctx.positions, table)
        if one:
            ops().attention_decode_qkv(rows, qw, kw, 1e-5, freq, k, v, out, *tail, H, 0.125, None, max(lens), write_kv=brings,
                                       rule=rule, magnitude=magnitude, whole=over == "projection", interleaved=interleaved, **more)
        else:
            q = torch.empty(R, H, D, dtype=torch.bfloat16, device=DEV)
            where = (ctx.positions, ctx.row_of_token, table if brings else None, page, q, k if brings else None,
                     v if brings else None, H, Hk if brings else 0, D)
            if row_store:
                ops().qk_row_norm_rope_store(rows, qw, qw if kw is None else kw, over if qw is not None else None, 1e-5, freq, magnitude,
                                             *where, D, v_transposed=True, interleaved=interleaved)
            else:
                ops().qk_norm_rope_store(rows, qw, kw, 1e-5, freq, *where, v_transposed=True, interleaved=interleaved)
            ops().attention_decode(q, k, v, out, *tail, 0.125, None, max(lens), exact=True, rule=rule)
        got.append([t.cpu().float() for t in (out, k, v)])
    return got


def _same(one, two):
    for a, b in zip(one, two):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


@pytest.mark.parametrize("H,Hk", [(8, 2), (32, 16)])
def test_norms_over_rows_whose_squares_leave_float32(H, Hk):
    """A row whose sum of squares overflows has a scale of exactly zero: zeros, and not every head normed by itself; an infinity
    gives NaN where it stands. In queries, and in the keys that are stored."""
    D, lens = 64, (40, 300, 64, 257)
    rows = rnd(len(lens), (H + 2 * Hk) * D, seed=3)
    rows[0, 5] = 3e19                                    # (its square is past 3.4e38)
    rows[1, 70] = float("inf")
    rows[2, H * D + 9] = -2e30
    rows[3, H * D + D + 1] = float("-inf")
    qw, kw = (1 + 0.1 * rnd(H * D, seed=4)).to(DEV), (1 + 0.1 * rnd(Hk * D, seed=5)).to(DEV)
    one, two = _one_and_two_launches(rows.to(DEV), H, Hk, qw, kw, torch.linspace(1.0, 0.01, 32, device=DEV), "projection", lens)
    _same(one, two)


@pytest.mark.parametrize("key_weight", [1, 4, None])
def test_rows_of_queries_alone_read_no_key_weight(key_weight):
    """Another layer's cache: whatever stands in the key weight's place (here shorter than a head, or the query weight) is not read."""
    H, Hk, D, lens = 16, 8, 64, (1, 33, 256, 300)
    rows = rnd(len(lens), H * D, seed=3).to(DEV)
    qw = (1 + 0.1 * rnd(H * D, seed=4)).to(DEV)
    kw = qw if key_weight is None else torch.full((key_weight,), float("nan"), device=DEV)
    one, _ = _one_and_two_launches(rows, H, Hk, qw, kw, torch.linspace(1.0, 0.01, 32, device=DEV), "projection", lens, brings=False)
    _, two = _one_and_two_launches(rows, H, Hk, qw, qw, torch.linspace(1.0, 0.01, 32, device=DEV), "projection", lens, brings=False)
    assert bool(torch.isfinite(two[0]).all())
    _same(one, two)


@pytest.mark.parametrize("H,Hk", [(8, 2), (20, 1), (32, 16)])
@pytest.mark.parametrize("brings,gated,magnitude", [(True, False, 1.0), (True, True, 1.0), (True, False, 1.2), (False, False, 1.0),
                                                    (False, False, 1.2)])
@pytest.mark.parametrize("normed,turned,interleaved", [(True, True, False), (True, True, True), (True, False, False),
                                                       (False, True, False), (False, False, False)])
def test_norms_a_head_have_the_bits_of_the_launch_they_stand_for(H, Hk, brings, gated, magnitude, normed, turned, interleaved):
    """Queries, the stored keys and the results, bit for bit, also without norms and without a rotation: the launch adds a head's
    squares in the order of the one that steps of more rows take, which depends on gates and magnitudes."""
    # (another order changes the last bit of a third of the sums, and that turns one rounding to bfloat16 in 60,000: many rows)
    D, lens = 64, (1, 2, 32, 33, 256, 257, 300, 513) + 24 * tuple(range(1, 41))
    rows = rnd(len(lens), (H + (2 * Hk if brings else 0)) * D + ((H + 7) // 8 * 8 if gated else 0), seed=3).to(DEV)
    qw, kw = ((1 + 0.1 * rnd(D, seed=4)).to(DEV), (1 + 0.1 * rnd(D, seed=5)).to(DEV)) if normed else (None, None)
    freq = torch.linspace(1.0, 0.01, D // 2, device=DEV) if turned else None
    one, two = _one_and_two_launches(rows, H, Hk, qw, kw, freq, "head", lens, brings, magnitude, gated, interleaved)
    assert bool(torch.isfinite(two[0]).all())
    _same(one, two)

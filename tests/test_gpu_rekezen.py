"""The Rekezen design in the engine against the plain implementation (tests/plain_rekezen.py): each mechanism's kernels
alone, whole prompts, stepwise decoding, portions down to two tokens, mixed batches on a pool at the schedule's peak with
slots used again, long decoding, first tokens, other sizes and constants, a token far away singled out by one score in
prompts and in decoding, generation through the entry point and the trace replay program.

float32 runs are held to the plain implementation with routers that read their input. Under bfloat16 a near-tie of a
router may fall the other way, which is no fault, so bfloat16 runs are held to their bound at every row with routers
whose choice hangs on their biases, and once with the drawn routers at most rows."""
import copy
import json
import math
import os
import random
import subprocess

import numpy as np
import pytest
import torch

import plain_rekezen as plain
from conftest import ROOT, prompt_tokens
from gpu_helpers import hand_context, make_engine, mixed_schedule, peak_pages, step_all
from rekezen_models import CONFIGS, finder, random_weights, write_model
from tolerances import bound, check_logits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FLIPS = 0.15          # share of rows that may miss the bfloat16 bound after a router's near-tie went the other way


class Yardstick:
    """The plain implementation in float64, and per row how far rounding moves the plain statement itself: in float32
    throughout, or with what every sublayer reads rounded to bfloat16. A row is held to the general bound or to three
    times that, whichever is larger."""

    def __init__(self, model_dir):
        self.exact, self.single = plain.PlainRekezen(model_dir), plain.PlainRekezen(model_dir, torch.float32)
        self._memo, self._noise = {}, {}

    def logits(self, tokens):
        key = tuple(tokens)
        if key not in self._memo:
            self._memo[key] = self.exact.logits(tokens)
        return self._memo[key]

    def noise(self, tokens, dtype="float32"):
        key = (tuple(tokens), dtype)
        if key not in self._noise:
            ref = self.logits(tokens)
            low = self.single.logits(tokens) if dtype == "float32" else self.exact.logits(tokens, inputs_as=torch.bfloat16)
            self._noise[key] = (low - ref).abs().max(dim=-1).values / float(ref.abs().max())
        return self._noise[key]


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    """(name, dtype) -> (folder, Yardstick): routers that read their input in float32, steady ones in bfloat16."""
    out = {}
    for name, (cfg, seed) in CONFIGS.items():
        for dtype in ("float32", "bfloat16"):
            d = write_model(cfg, seed, str(tmp_path_factory.mktemp(f"rekezen_{name}_{dtype}")), steady=dtype == "bfloat16")
            out[name, dtype] = (d, Yardstick(d))
    return out


def depth(name):
    return len(CONFIGS[name][0]["layers"])


def vocab(name):
    return CONFIGS[name][0]["vocab"]


def check(got, ref, what, rel, noise):
    """Every row within `rel` of the largest reference logit, or within three times its `noise` (Yardstick)."""
    got, ref = got.float().cpu(), ref.float().cpu()
    assert got.shape == ref.shape and torch.isfinite(got).all(), what
    row_err = (got - ref).abs().max(dim=-1).values / float(ref.abs().max())
    allowed = torch.maximum(torch.full_like(row_err, rel), 3.0 * noise[:row_err.shape[0]].float())
    over = (row_err > allowed).nonzero().flatten()
    assert over.numel() == 0, (f"{what}: row {int(over[0])} misses by {float(row_err[over[0]]):.3g}, allowed "
                               f"{float(allowed[over[0]]):.3g}; {over.numel()} of {got.shape[0]} rows")


def dev(t, dtype=torch.float32):
    return t.to(device=DEV, dtype=dtype).contiguous()


def i32(a):
    return torch.tensor(np.asarray(a, dtype=np.int32), device=DEV)


def near(got, want, rel, what=""):
    got, want = got.double().cpu(), want.double().cpu()
    assert got.shape == want.shape and torch.isfinite(got).all(), what
    assert float((got - want).abs().max()) <= rel * max(float(want.abs().max()), 1e-30), \
        f"{what}: {float((got - want).abs().max()):.3e} against {rel * float(want.abs().max()):.3e}"


# ------------------------------------------------------------------ the embedding
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E,buckets,mul_prev,mul_cur", [(64, 61, 31, 5), (37, 1, 7, 9), (1100, 5000, 1000003, 998244353), (8, 3, 0, 1),
                                                        (16, 1000, 3, 0)])
def test_second_table_over_segments_in_used_slots(E, buckets, mul_prev, mul_cur, dtype):
    """Three requests in slots that held other tokens, fed in segments of one token and more: every token's row is the
    one of its pair, also where the pair is cut between steps; a call that does not move the state on changes nothing."""
    from imparo_amd.kernels import ops
    g = torch.Generator().manual_seed(E)
    V = 90
    table, second = torch.randn(V, E, generator=g).to(dtype), torch.randn(buckets + 1, E, generator=g).to(dtype)
    slots, cuts = [4, 0, 2], [[1, 1, 5, 1], [2, 3, 1, 2], [7, 1, 1, 1]]
    state = i32([[11], [22], [33], [44], [55]])
    prompts = [prompt_tokens(V, sum(c), 5 + i) for i, c in enumerate(cuts)]
    fed = [0, 0, 0]
    for step in range(4):
        segs = [(fed[r], cuts[r][step]) for r in range(3)]
        ctx = hand_context(segs, 16, 4, torch.float32, torch.device(DEV), slots=slots, tables=[[0, 1]] * 3)
        ids = [t for r, (p0, n) in enumerate(segs) for t in prompts[r][p0:p0 + n]]
        want = []
        for r, (p0, n) in enumerate(segs):
            rows = plain.bigram_rows(prompts[r], buckets, mul_prev, mul_cur)[p0:p0 + n]
            want.append(0.6 * table[prompts[r][p0:p0 + n]].double() + second[rows].double())
        before = state.clone()
        for last in (False, True):
            out = torch.empty(len(ids), E, device=DEV)
            ops.embed_bigram(dev(table, dtype), dev(second, dtype), i32(ids), ctx.positions, ctx.row_of_token, ctx.seg_start,
                             ctx.seg_len, ctx.slot, state, out, mul_prev, mul_cur, 0.6, advance=last)
            near(out, torch.cat(want), 1e-6, f"step {step}")
            assert last or torch.equal(state, before)
        for r in range(3):
            fed[r] += cuts[r][step]
        assert [int(state[s]) for s in slots] == [p[f - 1] for p, f in zip(prompts, fed)]
        assert int(state[1]) == 22 and int(state[3]) == 44


# ------------------------------------------------------------------ streams and the norms that read them
def plain_norm(u, kind, w, b, eps):
    if kind == "layer":
        return plain.layer_norm(u, {"n": w, "n.b": b}, "n", eps)
    return plain.unit_rms(u, eps) * w + b if kind == "rms" else u * w + b


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("S,T,E", [(1, 5, 64), (2, 9, 37), (3, 70, 1024), (4, 3, 320), (4, 33, 4100), (5, 1, 1), (8, 6, 2048),
                                   (9, 4, 48), (16, 3, 1030), (4, 2, 16384), (3, 2, 16383)])
def test_streams_are_mixed_added_read_and_normed(S, T, E, out_dtype):
    """Every kind of norm; nothing pending, one delta, slices, experts' rows, those beside slices; copies apart or equal
    still; written back or for chosen rows only."""
    from imparo_amd.kernels import ops
    from imparo_amd.parts.base import RowsToCombine
    g = torch.Generator().manual_seed(S * 100 + E)
    r = lambda *shape: torch.randn(*shape, generator=g)
    X, w, b, eps = 2.0 * r(T, S, E) + 0.7, r(E), r(E), 1e-3
    mix, join, read = r(S, S) / math.sqrt(S), r(S), r(S)
    top = 3
    one, many, y, wt = r(T, E), r(6, T, E), r(T * top, E), torch.rand(T, top, generator=g)
    slot = torch.randperm(T * top, generator=g)
    choice = torch.randint(0, 9, (T, top), generator=g)
    experts = (wt.double()[:, :, None] * y.double()[slot].reshape(T, top, E)).sum(1)
    rows_of = lambda extra: RowsToCombine(dev(y), dev(one), i32(choice), dev(wt), i32(slot), 9, extra)
    rel = 3e-5 if out_dtype == torch.float32 else 6e-3
    cases = [(None, None), (dev(one), one.double()), (dev(many), many.double().sum(0)), (rows_of(None), experts),
             (rows_of(dev(many)), experts + many.double().sum(0)), (rows_of(dev(one)), experts + one.double())]
    for n, (delta, total) in enumerate(cases):
        kind = ("layer", "rms", "none")[n % 3] if n else "layer"
        for equal in (False, True):
            old = X[:, :1] if equal else X
            full = old.double().expand(T, S, E).permute(1, 0, 2)
            new = full if total is None else plain.spread_streams(full, total, mix.double(), join.double())
            want = plain_norm(plain.gather_streams(new, read.double()), kind, w.double(), b.double(), eps)
            links = dict(read=dev(read)) if total is None else dict(read=dev(read), mix=dev(mix), join=dev(join))
            x, out = dev(old[:, 0] if equal else old), torch.empty(T, E, dtype=out_dtype, device=DEV)
            moved = None if total is None else torch.full((T, S, E), 9.0, device=DEV) if equal else x if S > 1 else x.clone()
            ops.stream_norm(x, kind, dev(w), dev(b), eps, out, delta=delta, x_out=moved, **links)
            near(out.float(), want, rel, f"{n} {equal}")
            if total is not None:
                near(moved, new.permute(1, 0, 2), 3e-6, f"{n} {equal} copies")
            pick = [T - 1, 0, T // 2]
            x, out = dev(old[:, 0] if equal else old), torch.empty(3, E, dtype=out_dtype, device=DEV)
            links.pop("read")
            want = plain_norm(new.sum(0), kind, w.double(), b.double(), eps)[pick]
            ops.stream_norm(x, kind, dev(w), dev(b), eps, out, delta=delta, rows=i32(pick), streams=S, **links)
            near(out.float(), want, rel, f"{n} {equal} rows")
            assert torch.equal(x.cpu(), old[:, 0] if equal else old)


def test_norms_on_copies_of_a_stream():
    """The norm parts with a link before and behind them: both kinds of norm mix, read and move the copies on."""
    from imparo_amd.config.plan import PartSpec
    from imparo_amd.parts import part_class
    from imparo_amd.parts.base import Residual
    g = torch.Generator().manual_seed(3)
    T, E, S = 7, 48, 3
    r = lambda *shape: torch.randn(*shape, generator=g)
    x, delta, later = r(T, E), r(2, T, E), r(T, E)
    t = {"n": 0.5 + torch.rand(E, generator=g), "n.b": r(E)}
    links = []
    for i in range(2):
        t.update({f"c{i}.in": r(S), f"c{i}.out": r(S), f"c{i}.mix": r(S, S)})
        links.append(part_class("link", "hyper_connection")(PartSpec("hyper_connection", f"c{i}", dict(streams=S)), t, torch.device(DEV),
                                                          torch.float32))
    d = {k: v.double() for k, v in t.items()}
    ctx = hand_context([(0, T)], 16, 2, torch.float32, torch.device(DEV))
    for kind in ("layer_norm", "rms_norm"):
        def fn(u):
            return plain.layer_norm(u, d, "n", 1e-5) if kind == "layer_norm" else plain.unit_rms(u, 1e-5) * d["n"]
        part = part_class("norm", kind)(PartSpec(kind, "", dict(width=E, eps=1e-5, tensor="n")), t, torch.device(DEV), torch.float32)
        res = Residual(dev(x))
        near(part.forward_linked(ctx, res, links[0], torch.float32), fn(plain.gather_streams(x.double().expand(S, T, E), d["c0.in"])), 3e-6)
        res.pending, res.link = dev(delta), links[0]
        X = plain.spread_streams(x.double().expand(S, T, E), delta.double().sum(0), d["c0.mix"], d["c0.out"])
        near(part.forward_linked(ctx, res, links[1], torch.float32), fn(plain.gather_streams(X, d["c1.in"])), 1e-5)
        assert res.pending is None and res.link is None
        near(res.streams, X.permute(1, 0, 2), 3e-6)
        res.pending, res.link = dev(later), links[1]
        X2 = plain.spread_streams(X, later.double(), d["c1.mix"], d["c1.out"])
        near(part.forward_rows(ctx, res, i32([4, 1]), torch.float32), fn(X2.sum(0))[[4, 1]], 1e-5)
        near(res.streams, X.permute(1, 0, 2), 3e-6)
        res.pending = (dev(later), dev(later))
        with pytest.raises(ValueError):
            part.forward_linked(ctx, res, links[0], torch.float32)


# ------------------------------------------------------------------ norm, rotation, cache
ROWS = [  # heads, kv_heads, head_dim, value_dim, page, n_freq, extra columns
    (4, 2, 16, 16, 16, 8, 8), (6, 3, 64, 64, 64, 16, 2), (3, 1, 20, 12, 8, 10, 5), (8, 2, 128, 128, 64, 16, 8), (1, 1, 5, 7, 16, 2, 0),
    (5, 0, 32, 32, 16, 4, 3), (2, 2, 512, 300, 16, 256, 4), (20, 1, 80, 80, 16, 0, 4),
    (96, 8, 128, 64, 16, 32, 4)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("norm", [None, "head", "projection"])
@pytest.mark.parametrize("H,G,D,Dv,page,n_freq,extra", ROWS)
def test_norm_over_a_projection_rotation_and_store(H, G, D, Dv, page, n_freq, extra, norm, dtype):
    """Few tokens (several blocks a token) and many, pairs in halves and neighbouring, sine and cosine times a constant,
    values transposed inside a page or not, queries alone, rows that go on behind the values."""
    from imparo_amd.kernels import ops
    eps, magnitude = 1e-3, 1.37
    for segs, interleaved, vt in (([(3, 1), (0, 9), (page - 1, 2)], False, True), ([(0, 70), (5, 1)], True, False), ([(30, 260)], False, False)):
        g = torch.Generator().manual_seed(H + D + len(segs))
        T = sum(n for _, n in segs)
        width = (H + G) * D + G * Dv
        rows = torch.randn(T, width + extra, generator=g)
        wq, wk = torch.randn(H * D, generator=g), torch.randn(G * D, generator=g)
        if norm == "head":
            wq, wk = wq[:D], wk[:D] if G else wk
        freq = 1.0 / torch.arange(1, n_freq + 1).float()
        n_pages = sum((p0 + n + page - 1) // page for p0, n in segs) + 1
        ctx = hand_context(segs, page, n_pages, dtype, torch.device(DEV))
        q = torch.empty(T, H, D, dtype=dtype, device=DEV)
        kc = torch.zeros(n_pages, max(G, 1), page, D, dtype=dtype, device=DEV)
        vc = torch.zeros((n_pages, max(G, 1), Dv, page) if vt else (n_pages, max(G, 1), page, Dv), dtype=dtype, device=DEV)
        ops.qk_row_norm_rope_store(dev(rows), dev(wq) if norm else None, dev(wk) if norm and G else None, norm, eps, dev(freq) if n_freq else None,
                                   magnitude, ctx.positions, ctx.row_of_token, ctx.block_tables[0] if G else None, page, q,
                                   kc if G else None, vc if G else None, H, G, D, Dv, v_transposed=vt, interleaved=interleaved)
        pos = ctx.positions.cpu()

        def plain_side(x, n, w):
            x = x.double()
            if norm == "projection":
                x = plain.unit_rms(x, eps) * w
            x = x.reshape(T, n, D)
            if norm == "head":
                x = plain.unit_rms(x, eps) * w
            a = (pos.double()[:, None] * freq.double()[None])[:, None, :]
            c, s = torch.cos(a) * magnitude, torch.sin(a) * magnitude
            y = x.clone()
            u, v = (slice(0, 2 * n_freq, 2), slice(1, 2 * n_freq, 2)) if interleaved else (slice(0, n_freq), slice(n_freq, 2 * n_freq))
            y[..., u], y[..., v] = x[..., u] * c - x[..., v] * s, x[..., v] * c + x[..., u] * s
            return y
        rel = 5e-6 if dtype == torch.float32 else 6e-3
        near(q.float(), plain_side(rows[:, :H * D], H, wq), rel, "q")
        if not G:
            continue
        table, row_of = ctx.block_tables[0].cpu(), ctx.row_of_token.cpu()
        at = [(int(table[row_of[t], pos[t] // page]), int(pos[t]) % page) for t in range(T)]
        got_k = torch.stack([kc[p, :, s] for p, s in at]).float()
        got_v = torch.stack([vc[p, :, :, s] if vt else vc[p, :, s] for p, s in at]).float()
        near(got_k, plain_side(rows[:, H * D:(H + G) * D], G, wk), rel, "k")
        near(got_v, rows[:, (H + G) * D:width].reshape(T, G, Dv), rel, "v")
        touched = torch.zeros(n_pages, page, dtype=torch.bool)
        for p, s in at:
            touched[p, s] = True
        assert float(kc.permute(0, 2, 1, 3)[~touched.to(DEV)].abs().max()) == 0.0


# ------------------------------------------------------------------ attention with a gate a head
def gated_case(H, G, D, V, segments, page, dtype, cap=None, boost=None, seed=0, kernel="wave", parts=None, drop=None):
    """q, k, v for rows given as (start, tokens) whose earlier positions are in the cache; pages in a shuffled order;
    everything in the cache that is no key of a row is not a number. -> (kernel output [tokens, H * V], plain output).
    `boost` (row, key position): that key matches the row's last query. `drop`: the plain statement without that key."""
    from imparo_amd.kernels import ops
    g = torch.Generator().manual_seed(seed + D + V)
    bf = (lambda t: t.to(torch.bfloat16).float()) if dtype == torch.bfloat16 else (lambda t: t)
    scale, nan = 1.0 / math.sqrt(D), float("nan")
    n_pages = sum((p0 + n + page - 1) // page for p0, n in segments) + 3
    order = [p for p in torch.randperm(n_pages, generator=g).tolist() if p != 0]
    kc, vc = torch.full((n_pages, G, page, D), nan), torch.full((n_pages, G, page, V), nan)
    q_all, ref_all, tables, gates = [], [], [], []
    for r, (p0, n) in enumerate(segments):
        L = p0 + n
        q, k, v = bf(torch.randn(L, H, D, generator=g)), bf(torch.randn(L, G, D, generator=g)), bf(torch.randn(L, G, V, generator=g))
        z = 2.0 * torch.randn(L, H, generator=g)
        if boost is not None and boost[0] == r:
            k[boost[1]] = bf(q[L - 1, ::H // G] * 3.0)
        pos = torch.arange(L)
        seen = pos[None, :] <= pos[:, None]
        if drop is not None and r == 0:
            seen[L - 1, drop] = False
        o = plain.capped_attention(q.double(), k.double(), v.double(), seen, scale, cap)
        ref_all.append(plain.gate_heads(o, z.double()).reshape(L, H * V)[p0:].float())
        q_all.append(q[p0:])
        gates.append(z[p0:])
        tables.append([order.pop() for _ in range((L + page - 1) // page)])
        for p in range(L):
            kc[tables[-1][p // page], :, p % page], vc[tables[-1][p // page], :, p % page] = k[p], v[p]
    ctx = hand_context(segments, page, n_pages, dtype, torch.device(DEV), tables=tables)
    q = dev(torch.cat(q_all), dtype)
    T = q.shape[0]
    out = torch.empty(T, H * V, dtype=dtype, device=DEV)
    rows = dev(torch.cat([torch.full((T, 5), nan), torch.cat(gates), torch.full((T, 3), nan)], dim=1))
    rule = ops.attention_rule(H, softcap=cap).with_gate(rows, 5)
    if kernel == "wave":
        ops.attention(q, dev(kc, dtype), dev(vc, dtype), out, ctx.positions, ctx.row_of_token, ctx.block_tables[0], scale, None, rule=rule)
        return out.float().cpu(), torch.cat(ref_all)
    kd, vd = dev(kc, dtype), dev(vc.permute(0, 1, 3, 2), dtype)
    if ctx.n_single_rows:
        splits = (ctx.max_context + ops.decode_split() - 1) // ops.decode_split()
        part_o = torch.full((ctx.n_single_rows * H * splits * D,), nan, device=DEV)
        part_ml = torch.full((ctx.n_single_rows * H * splits * 2,), nan, device=DEV)
        ops.attention_decode(q, kd, vd, out, part_o, part_ml, ctx.single_rows, ctx.n_single_rows, ctx.seg_start, ctx.positions,
                             ctx.block_tables[0], scale, None, ctx.max_context, exact=True, rule=rule)
    if ctx.n_portion_rows:
        tiles = sum((n + 63) // 64 for n in ctx.host_seg_len if n > 1)
        part_o = part_ml = None
        if parts:
            part_o = torch.full((T * H * parts * D,), nan, device=DEV)
            part_ml = torch.full((T * H * parts * 2,), nan, device=DEV)
        ops.attention_prefill(q, kd, vd, out, ctx.portion_rows, ctx.n_portion_rows, tiles, ctx.seg_start, ctx.seg_len, ctx.positions,
                              ctx.block_tables[0], scale, None, part_o, part_ml, parts or 1, exact=True, rule=rule)
    return out.float().cpu(), torch.cat(ref_all)


@pytest.mark.parametrize("cap", [None, 2.0, 30.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,V,page", [(4, 2, 16, 32, 16), (3, 1, 24, 40, 64), (2, 1, 12, 20, 8)])
def test_a_gate_a_head(H, G, D, V, page, dtype, cap):
    got, ref = gated_case(H, G, D, V, [(150, 37), (299, 1), (0, 70), (63, 1), (0, 1)], page, dtype, cap)
    near(got, ref, 3e-6 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("cap", [None, 2.0])
@pytest.mark.parametrize("H,G,D,page", [(4, 2, 16, 16), (8, 2, 64, 64), (2, 2, 128, 32), (3, 1, 48, 64), (20, 1, 80, 16), (40, 2, 64, 128)])
def test_a_gate_a_head_on_the_matrix_cores(H, G, D, page, cap):
    """Decoding over one split of the keys and several, the prompt kernels for head sizes in steps of 32 and of 16."""
    got, ref = gated_case(H, G, D, D, [(150, 37), (299, 1), (0, 70), (700, 1), (63, 1), (0, 1), (500, 130)], page, torch.bfloat16, cap,
                          kernel="mfma")
    near(got, ref, 1e-2)
    got, ref = gated_case(H, G, D, D, [(100, 1), (40, 1)], page, torch.bfloat16, cap, kernel="mfma")
    near(got, ref, 1e-2)


@pytest.mark.parametrize("parts", [2, 5])
def test_a_gate_a_head_over_keys_in_parts(parts):
    got, ref = gated_case(8, 2, 64, 64, [(400, 90), (0, 20), (130, 64)], 64, torch.bfloat16, 9.0, kernel="mfma", parts=parts)
    near(got, ref, 1e-2)


@pytest.mark.parametrize("kernel,dtype", [("wave", torch.float32), ("wave", torch.bfloat16), ("mfma", torch.bfloat16)])
@pytest.mark.parametrize("n_last", [1, 5, 70])
def test_a_far_key_among_hundreds(kernel, dtype, n_last):
    """One key, the first of all, far back, at both sides of a page's border or right before the query, outweighs the rest."""
    L, tol = 1150, 3e-6 if dtype == torch.float32 else 1e-2
    for key in (0, 47, 63, 64, 255, 256, L - 2):
        args = dict(cap=30.0, boost=(0, key), seed=key, kernel=kernel)
        got, ref = gated_case(4, 2, 64, 64, [(L - n_last, n_last), (3, 1)], 64, dtype, **args)
        near(got, ref, tol, f"key {key}")
    wrong = gated_case(4, 2, 64, 64, [(L - n_last, n_last), (3, 1)], 64, dtype, drop=L - 2, **args)[1]
    assert float((wrong[n_last - 1] - ref[n_last - 1]).abs().max()) > 0.2 * float(ref[n_last - 1].abs().max())


# ------------------------------------------------------------------ experts
@pytest.mark.parametrize("T", [3, 40, 100])
@pytest.mark.parametrize("X,top", [(1, 1), (5, 5), (12, 4), (64, 16), (200, 3), (512, 8)])
def test_weights_over_the_chosen_outputs(X, top, T):
    """The largest outputs are chosen, weighed by a softmax over themselves, however far below the largest they lie."""
    from imparo_amd.kernels import ops
    g = torch.Generator().manual_seed(X + T)
    z = torch.stack([torch.randperm(X, generator=g) for _ in range(T)]).float() * 0.37 - 4.0
    z[T // 2] *= 400.0 / X                       # outputs so far apart that a softmax over all of them would lose the rest
    best, want = torch.topk(z.double(), top, dim=-1)
    for always in (0, 1, 3):
        choice, weight = torch.empty(T, top + always, dtype=torch.int32, device=DEV), torch.empty(T, top + always, device=DEV)
        ops.moe_route(dev(z), None, choice, weight, top, scoring="chosen", scale=1.5, always=always)
        assert torch.equal(choice.cpu().long()[:, :top], want)
        near(weight[:, :top], 1.5 * torch.softmax(best, dim=-1), 2e-6)
        assert torch.equal(choice.cpu()[:, top:], (X + torch.arange(always, dtype=torch.int32)).expand(T, always))
        assert bool((weight[:, top:] == 1.0).all())
    if T <= ops.moe_route_plan_tokens():
        rows = ops.moe_tile_rows(T * top, X, torch.bfloat16)
        n = T * (top + 1)
        tiles = torch.empty(ops.moe_max_tiles(n, X + 1, rows), 3, dtype=torch.int32, device=DEV)
        s1, s2 = torch.empty(n, dtype=torch.int32, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV)
        choice, weight = torch.empty(T, top + 1, dtype=torch.int32, device=DEV), torch.empty(T, top + 1, device=DEV)
        ops.moe_route_plan(dev(z), None, choice, weight, top, X + 1, rows, s1, s2, tiles, scoring="chosen", always=1)
        assert torch.equal(choice.cpu().long()[:, :top], want)
        near(weight[:, :top], torch.softmax(best, dim=-1), 2e-6)
        assert sorted(s1.cpu().tolist()) == list(range(n)) and bool((choice.cpu()[s2.cpu().long() // (top + 1), top] == X).all())


@pytest.mark.parametrize("S,E,T", [(1, 2048, 1200), (2, 1028, 2001), (4, 1024, 2500), (8, 2048, 520), (2, 1028, 3500), (4, 1024, 4200), (2, 256, 33000)])
@pytest.mark.parametrize("n_delta", [1, 2, 3])
@pytest.mark.parametrize("norm", ["layer", "none"])
def test_streams_of_many_rows_are_those_of_few(S, E, T, n_delta, norm):
    """From some rows on a block asks for a row where it uses it, and not ahead: the same bits as in thirds of the rows, the copies
    that are written back and the normed rows."""
    from imparo_amd.kernels import ops
    g = torch.Generator().manual_seed(S)
    r = lambda *shape: dev(torch.randn(*shape, generator=g))
    x, delta, w, b, mix, join, read = r(T, S, E), r(n_delta, T, E), r(E), r(E), r(S, S), r(S), r(S)

    def run(lo, hi):
        x_out, out = torch.empty(hi - lo, S, E, device=DEV), torch.empty(hi - lo, E, device=DEV)
        weights = (w, b) if norm != "none" else (None, None)
        ops.stream_norm(x[lo:hi], norm, *weights, 1e-5, out, delta=delta[:, lo:hi].contiguous(), mix=mix, join=join, read=read, x_out=x_out)
        return x_out, out

    many, thirds = run(0, T), [run(T * i // 3, T * (i + 1) // 3) for i in range(3)]
    for i in range(2):
        assert torch.equal(many[i], torch.cat([part[i] for part in thirds]))


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid", "chosen"])
@pytest.mark.parametrize("X,top", [(1, 1), (8, 4), (16, 16), (32, 1), (33, 1), (33, 3), (64, 2), (63, 5), (64, 16)])
def test_choice_among_few_outputs_is_the_general_one(X, top, scoring):
    """At most 64 outputs are ranked by counting; the same rows with outputs past the 64th that cannot be chosen go the
    general way and give the same choices and weights, bit for bit: equal outputs, rows with too few that can be chosen
    (minus infinity, NaN), and infinity. The plan made in the same launch holds every chosen entry once."""
    from imparo_amd.kernels import ops
    T, wide = 40, 65
    z = torch.randn(T, X, generator=torch.Generator().manual_seed(X)) * 2
    z[1], z[2], z[3, 0], z[4, X // 2], z[5, X // 2:] = 0.5, z[2].round(), float("inf"), float("nan"), -float("inf")
    corr = (0.3 * torch.randn(X, generator=torch.Generator().manual_seed(top))).round(decimals=1)
    pad = lambda t: torch.cat([t, torch.full((*t.shape[:-1], wide - X), -float("inf"))], -1)
    got = []
    for logits, c in ((z, corr), (pad(z), pad(corr))):
        choice, weight = torch.empty(T, top, dtype=torch.int32, device=DEV), torch.empty(T, top, device=DEV)
        ops.moe_route(dev(logits), dev(c), choice, weight, top, scoring=scoring, normalize=True, scale=1.3)
        got.append((choice.cpu(), weight.cpu()))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1].view(torch.int32), got[1][1].view(torch.int32)) or \
        torch.equal(got[0][1].nan_to_num(7.0), got[1][1].nan_to_num(7.0))
    rows, n = ops.moe_tile_rows(T * top, X, torch.bfloat16), T * top
    tiles = torch.empty(ops.moe_max_tiles(n, X, rows), 3, dtype=torch.int32, device=DEV)
    s1, s2 = torch.empty(n, dtype=torch.int32, device=DEV), torch.full((n,), -1, dtype=torch.int32, device=DEV)
    ops.moe_route_plan(dev(z), dev(corr), choice, weight, top, X, rows, s1, s2, tiles, scoring=scoring, normalize=True, scale=1.3)
    assert torch.equal(choice.cpu(), got[0][0])
    e, slot = choice.cpu().flatten(), s1.cpu()
    real = e < X
    assert bool((slot[~real] == -1).all()) and sorted(slot[real].tolist()) == list(range(int(real.sum())))
    assert bool((e[s2.cpu()[:int(real.sum())].long()].diff() >= 0).all())          # an expert's slots lie together
    used = tiles.cpu()[tiles.cpu()[:, 0] >= 0]
    assert int(used[:, 2].sum()) == int(real.sum())


@pytest.mark.parametrize("n,half", [(7, 24), (5, 13), (900, 64)])
def test_gated_unit_with_bounds_over_experts_rows(n, half):
    from imparo_amd.kernels import ops
    gu = 3.0 * torch.randn(n, 2 * half, generator=torch.Generator().manual_seed(n))
    gen = torch.Generator().manual_seed(half)
    entry, choice = torch.randperm(n, generator=gen), torch.randint(0, 3, (n,), generator=gen)
    wt = torch.rand(n, generator=gen)
    for dt, rel in ((torch.float32, 3e-6), (torch.bfloat16, 5e-3)):
        for limits, alpha, weight in (((1.2, 0.3, 4.0), 1.702, None), ((7.0, 7.0, 7.0), 0.5, wt), (None, 1.0, wt), (None, 1.0, None)):
            g, u = gu[:, :half].double(), gu[:, half:].double()
            if weight is not None:
                g, u = g * weight[entry].double()[:, None], u * weight[entry].double()[:, None]
            if limits:
                lim = torch.tensor(limits).double()[choice[entry]][:, None]
                g, u = torch.minimum(g, lim), torch.maximum(torch.minimum(u, lim), -lim) + 1.0
            hidden = torch.empty(n, half, dtype=dt, device=DEV)
            ops.moe_gated(dev(gu), None if weight is None else dev(weight), i32(entry), hidden, i32(choice),
                          dev(torch.tensor(limits)) if limits else None, alpha)
            near(hidden.float(), g * torch.sigmoid(alpha * g) * u, rel)


@pytest.mark.parametrize("T,X,top,F,K", [(3, 5, 2, 32, 64), (20, 4, 2, 96, 200), (70, 3, 3, 64, 72), (600, 4, 2, 160, 512), (1, 1, 1, 32, 8)])
@pytest.mark.parametrize("bounds", [True, False])
def test_product_of_the_experts_with_the_unit_behind_it(T, X, top, F, K, bounds):
    """Gate and up rows in blocks of 32 in one product whose epilogue gates, for few rows an expert and many, with a bound
    for every expert and a factor on what a slot reads, or neither."""
    from imparo_amd.kernels import ops
    g = torch.Generator().manual_seed(T)
    h, n = torch.randn(T, K, generator=g).to(torch.bfloat16), T * top
    gate, up = ((torch.randn(X, F, K, generator=g) * 1.5 / math.sqrt(K)).to(torch.bfloat16) for _ in range(2))
    choice = torch.stack([torch.randperm(X, generator=g)[:top] for _ in range(T)])
    limits, wt = torch.rand(X, generator=g) + 0.3, torch.rand(T, top, generator=g) + 0.5
    rows = ops.moe_tile_rows(n, X, torch.bfloat16)
    slot, entry = torch.empty(n, dtype=torch.int32, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV)
    tiles = torch.empty(ops.moe_max_tiles(n, X, rows), 3, dtype=torch.int32, device=DEV)
    ops.moe_plan(i32(choice), X, rows, slot, entry, tiles)
    w = torch.stack([gate.view(X, F // 32, 32, K), up.view(X, F // 32, 32, K)], dim=2).reshape(X, 2 * F, K)
    hidden = torch.full((n, F), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.moe_gemm(dev(h, torch.bfloat16), dev(w, torch.bfloat16), hidden, tiles, rows, entry, gather_div=top, epilogue="gated",
                 limits=dev(limits) if bounds else None, alpha=1.702, weight=dev(wt).view(-1) if bounds else None)
    got = hidden.float().cpu()[slot.cpu().long()].view(T, top, F)
    for j in range(top):
        a = torch.einsum("tk,tfk->tf", h.double(), gate[choice[:, j]].double())
        b = torch.einsum("tk,tfk->tf", h.double(), up[choice[:, j]].double())
        if bounds:
            a, b, lim = a * wt[:, j:j + 1], b * wt[:, j:j + 1], limits[choice[:, j]].double()[:, None]
            a, b = torch.minimum(a, lim), torch.maximum(torch.minimum(b, lim), -lim) + 1.0
            want = a * torch.sigmoid(1.702 * a) * b
        else:
            want = a * torch.sigmoid(a) * b
        near(got[:, j], want, 8e-3, f"choice {j}")


@pytest.mark.parametrize("counts,N,K", [((128, 127, 129, 1, 0, 300), 256, 64), ((128, 127, 129, 1, 0, 300), 256, 128), ((200, 256), 500, 128), ((513, 100, 60), 448, 192),
                                        ((128, 128, 128), 768, 1024)])
@pytest.mark.parametrize("epilogue,out_dtype", [("relu2", torch.bfloat16), (None, torch.float32), ("gated", torch.bfloat16)])
def test_product_of_the_experts_at_the_edges_of_wide_tiles(counts, N, K, epilogue, out_dtype):
    """Tiles of 128 slots by 256 columns beside experts with a row more or less, none, or one; columns and K-steps beside
    whole tiles and rounds; with empty tiles in the list and without. Sums of K products of bfloat16 in float32."""
    from imparo_amd.kernels import ops
    N = N // 64 * 64 if epilogue == "gated" else N
    g = torch.Generator().manual_seed(N + K)
    X, n = len(counts), sum(counts)
    choice = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(n, generator=g)]
    h = torch.randn(n, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(X, N, K, generator=g) / math.sqrt(K)).to(torch.bfloat16)
    slot, entry = torch.empty(n, dtype=torch.int32, device=DEV), torch.empty(n, dtype=torch.int32, device=DEV)
    live = sum(-(-c // 128) for c in counts)
    tiles = torch.empty(ops.moe_max_tiles(n, X, 128), 3, dtype=torch.int32, device=DEV)
    ops.moe_plan(i32(choice), X, 128, slot, entry, tiles)
    for length in (tiles.shape[0], live + 1, live):
        tiles = tiles[:length].contiguous()
        assert (tiles[:, 0] >= 0).sum() == live and (length > live) == bool((tiles[-1, 0] < 0).item())
        cols = N // 2 if epilogue == "gated" else N
        out = torch.full((n, cols), 7.0, dtype=out_dtype, device=DEV)
        ops.moe_gemm(dev(h, torch.bfloat16), dev(w, torch.bfloat16), out, tiles, 128, entry, gather_div=1, epilogue=epilogue)
        z = torch.stack([h[i].double() @ w[int(choice[i])].double().t() for i in range(n)])
        if epilogue == "gated":
            z = z.view(n, N // 64, 2, 32)
            z = (z[:, :, 0] * torch.sigmoid(z[:, :, 0]) * z[:, :, 1]).reshape(n, cols)
        elif epilogue == "relu2":
            z = torch.relu(z).square()
        near(out.float().cpu()[slot.cpu().long()], z, 8e-3 if out_dtype == torch.bfloat16 else 1e-6 * math.sqrt(K))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 9, 70, 300])
@pytest.mark.parametrize("ff,shared_ff,E,X,top", [(24, 40, 64, 6, 2), (13, 9, 48, 3, 3), (64, None, 128, 16, 4), (16, 16, 36, 1, 1),
                                                  (100, 104, 96, 10, 8), (48, 48, 64, 5, 3)])
def test_routed_experts_with_a_shared_unit(ff, shared_ff, E, X, top, T, dtype):
    """The feed-forward part whole: as one result, and as rows left for the next launch to add."""
    from imparo_amd.config import plan_from_config
    from imparo_amd.parts import part_class
    from rekezen_models import attention, layer, moe
    mlp = moe(ff, 1.1, X, top, None if shared_ff is None else (shared_ff, 0.7))
    cfg = dict(architecture="Rekezen", vocab=10, width=E, norm=dict(eps=1e-5), layers=[layer(attention(1, 1, 8, 8), mlp)])
    w = {k: v.to(dtype) for k, v in random_weights(cfg, E + X, steady=True).items()}
    spec = plan_from_config(cfg)[1].layers[0].ffn
    part = part_class("feed_forward", spec.kind)(spec, w, torch.device(DEV), dtype)
    h = torch.randn(T, E, generator=torch.Generator().manual_seed(T)).to(part.in_dtype)
    want = plain.mixture(h.double(), {k: v.double() for k, v in w.items()}, "l0.mlp", mlp)
    ctx = hand_context([(0, T)], 16, 32, dtype, torch.device(DEV))
    tol = 3e-6 if dtype == torch.float32 else 1.2e-2
    near(part.forward(ctx, dev(h, h.dtype)), want, tol)
    r = part.forward_parts(ctx, dev(h, h.dtype))
    assert part.always == (shared_ff is not None and abs(shared_ff - ff) < 8) and (r.extra is None) == (part.always or shared_ff is None)
    y = (r.weight.double()[:, :, None] * r.y.double()[r.slot_of_entry.long()].view(T, top + part.always, E)).sum(1)
    if r.extra is not None:
        y = y + (r.extra.double().sum(0) if r.extra.dim() == 3 else r.extra.double())
    near(y, want, tol)


# ------------------------------------------------------------------ the model
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_whole_prompt_and_stepwise(models, name, dtype):
    """A prompt whole; then most of it whole and its last 50 tokens one by one (captured steps)."""
    from imparo_amd.engine import StepEntry
    d, y = models[name, dtype]
    tokens = prompt_tokens(vocab(name), 170, 7)
    ref, noise, rel = y.logits(tokens), y.noise(tokens, dtype), bound(dtype, depth(name))
    eng = make_engine(d, dtype)
    whole = eng.step([StepEntry("w", tokens, list(range(170)))]).cpu()
    eng.release("w")
    check(whole, ref, f"{name} whole", rel, noise)
    head = eng.step([StepEntry("d", tokens[:120], list(range(120)))]).cpu()
    tail = [eng.step([StepEntry("d", [t], [0])]).cpu() for t in tokens[120:]]
    eng.release("d")
    stepwise = torch.cat([head] + tail)
    check(stepwise, ref, f"{name} stepwise", rel, noise)
    if dtype == "float32":
        check(stepwise, whole, f"{name} stepwise against whole", 3e-6, noise)


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_every_layer_alone(name, tmp_path):
    """The model cut behind its first, second, ... layer: the first one that differs is named by the failing case."""
    from imparo_amd.engine import StepEntry
    cfg, seed = CONFIGS[name]
    tokens = prompt_tokens(cfg["vocab"], 40, 9)
    for k in range(1, len(cfg["layers"])):
        d = write_model(dict(cfg, layers=cfg["layers"][:k]), seed, str(tmp_path / f"cut{k}"))
        got = make_engine(d, "float32").step([StepEntry("a", tokens, list(range(40)))]).cpu()
        y = Yardstick(d)
        check(got, y.logits(tokens), f"{name}: {k} layers", bound("float32", k), y.noise(tokens))


@pytest.mark.parametrize("name", ["A", "C", "D"])
def test_drawn_routers_in_bfloat16(models, name):
    """Routers that read their input, in bfloat16: all but the rows whose choice a rounding turned."""
    from imparo_amd.engine import StepEntry
    d, y = models[name, "float32"]
    tokens = prompt_tokens(vocab(name), 300, 12)
    ref = y.logits(tokens)
    got = make_engine(d, "bfloat16").step([StepEntry("a", tokens, list(range(300)))]).cpu()
    err = (got - ref).abs().max(dim=-1).values / float(ref.abs().max())
    assert torch.isfinite(got).all() and float((err > bound("bfloat16", depth(name))).float().mean()) <= FLIPS


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name,page", [("A", 16), ("B", 8), ("C", 16), ("D", 64), ("E", 32)])
def test_portions_of_changing_size(models, name, page, dtype):
    """Portions down to two tokens, cut inside pages, also without captured steps."""
    d, y = models[name, dtype]
    tokens = prompt_tokens(vocab(name), 160, 8)
    ref, noise = y.logits(tokens), y.noise(tokens, dtype)
    for cuts, graphs in (((2, 3, 17, 2, 1, 31, 1, 1, 5), True), ((64, 2, 9), False), ((1,), True), ((2,), False)):
        eng = make_engine(d, dtype, page_size=page, use_graphs=graphs)
        got = step_all(eng, "p", tokens if len(cuts) > 1 else tokens[:45], cuts)
        check(got, ref[:got.shape[0]], f"{name} cuts {cuts}", bound(dtype, depth(name)), noise)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name,page", [("A", 8), ("B", 8), ("C", 16), ("D", 16), ("E", 16)])
def test_mixed_batches_on_a_full_pool(models, name, page, dtype):
    """Six unequal requests, at most four live, portions beside single tokens, on a pool of exactly the schedule's
    peak and four slots: pages and state slots are used again. Each request's logits are those it has alone."""
    from imparo_amd.engine import StepEntry
    d, y = models[name, dtype]
    lengths = [70, 33, 1, 90, 2, 51]
    prompts = [prompt_tokens(vocab(name), n, 20 + i) for i, n in enumerate(lengths)]
    steps = mixed_schedule(random.Random(5), lengths, max_live=4)
    eng = make_engine(d, dtype, page_size=page, max_tokens=peak_pages(steps, page) * page, max_requests=4)
    got = {i: [] for i in range(len(lengths))}
    for entries, ends in steps:
        out = eng.step([StepEntry(rid, prompts[rid][lo:hi], list(range(hi - lo))) for rid, lo, hi in entries]).cpu()
        at = 0
        for rid, lo, hi in entries:
            got[rid].append(out[at:at + hi - lo])
            at += hi - lo
        for rid in ends:
            eng.release(rid)
    for i, p in enumerate(prompts):
        check(torch.cat(got[i]), y.logits(p), f"{name} request {i}", bound(dtype, depth(name)), y.noise(p, dtype))
    eng.cache.check()
    assert eng.free_pages() == [g.pool.n_pages for g in eng.cache.groups]


@pytest.mark.parametrize("name", ["A", "D"])
def test_long_decoding_and_first_tokens(models, name):
    """One prompt token, then 330 single-token steps; and requests of one and of two tokens alone, in used slots."""
    from imparo_amd.engine import StepEntry
    tokens = prompt_tokens(vocab(name), 331, 3)
    for dtype in ("float32", "bfloat16"):
        d, y = models[name, dtype]
        exact, noise = y.logits(tokens), y.noise(tokens, dtype)
        eng = make_engine(d, dtype, page_size=16)
        got = torch.cat([eng.step([StepEntry("r", [t], [0])]).cpu() for t in tokens])
        check(got, exact, "long decoding", bound(dtype, depth(name)), noise)
        eng.release("r")
        two = eng.step([StepEntry("x", tokens[:1], [0]), StepEntry("y", tokens[:2], [0, 1])]).cpu()
        check(two, torch.cat([exact[:1], exact[:2]]), "first tokens", bound(dtype, depth(name)), torch.cat([noise[:1], noise[:2]]))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_token_far_back(tmp_path, dtype):
    """A token that the last one's queries look for, far back, at page borders, first of all, and right before it, in a
    prompt, in a portion and in decoding: through a layer of its own keys and one that reads them."""
    from imparo_amd.engine import StepEntry
    cfg, over = finder(3, 5)
    d = write_model(cfg, 9, str(tmp_path / "m"), overrides=over)
    y = Yardstick(d)
    L = 700
    base = [t if t not in (3, 5) else 7 for t in prompt_tokens(cfg["vocab"], L, 2)] + [3]
    nowhere = y.logits(base)
    eng = make_engine(d, dtype, page_size=64, max_tokens=4096)
    for at in (0, 1, 63, 64, 255, 256, 400, L - 1):
        tokens = list(base)
        tokens[at] = 5
        ref, noise = y.logits(tokens), y.noise(tokens, dtype)
        assert float((ref[-1] - nowhere[-1]).abs().max()) > 0.1 * float(ref.abs().max())
        rel = bound(dtype, 2)
        for n_last in (1, 2, 40, L + 1):
            if n_last <= L:
                eng.step([StepEntry(n_last, tokens[:-n_last], [])])
        out = eng.step([StepEntry(n, tokens[-n:], [n - 1]) for n in (1, 2, 40, L + 1)]).cpu()
        check(out, ref[-1:].expand(4, -1), f"token at {at}", rel, noise[-1:].expand(4))
        for n in (1, 2, 40, L + 1):
            eng.release(n)


def test_other_constants(models, tmp_path):
    """Values that a model may happen to make equal or 1: another eps, factor, multiplier, scale, cap, rotation, scaling,
    bound, number of experts chosen, source of keys or layer without feed-forward moves the logits, and by what the plain
    implementation says."""
    from imparo_amd.engine import StepEntry
    from imparo_amd.weights.safetensors_io import save_file
    cfg, seed = CONFIGS["A"]
    tokens = prompt_tokens(cfg["vocab"], 60, 4)
    base = make_engine(models["A", "float32"][0], "float32").step([StepEntry("a", tokens, list(range(60)))]).cpu()
    m = lambda c, i=0: c["layers"][i]["mixer"]
    f = lambda c, i=0: c["layers"][i]["mlp"]
    changes = [
        lambda c: c["norm"].update(eps=1e-1),
        lambda c: c.update(logit_scale=-1.5),
        lambda c: c.pop("logit_scale"),
        lambda c: c["embedding"]["bigram"].update(mul_prev=8),
        lambda c: c["embedding"]["bigram"].update(mul_cur=0),
        lambda c: m(c).update(scale=1.3),
        lambda c: m(c, 1).update(softcap=0.5),
        lambda c: m(c).pop("softcap"),
        lambda c: m(c)["rot"].update(base=33.0),
        lambda c: m(c)["rot"].update(dims=4),
        lambda c: m(c).pop("rot"),
        lambda c: m(c)["rot"].pop("scaling"),
        lambda c: m(c)["rot"]["scaling"].update(factor=9.0),
        lambda c: m(c)["rot"]["scaling"].update(original=700),
        lambda c: m(c)["rot"]["scaling"].update(fast=2.0),
        lambda c: m(c)["rot"]["scaling"].update(slow=5.0),
        lambda c: m(c, 1)["rot"].pop("scaling"),
        lambda c: f(c)["expert"].update(limit=0.3),
        lambda c: f(c)["shared"].update(limit=0.2),
        lambda c: f(c)["router"].update(top=6),
        lambda c: f(c)["router"].update(top=1),
        lambda c: c["layers"][0].update(mlp=None),
        lambda c: c.pop("streams"),
        lambda c: f(c).pop("shared"),
        lambda c: c.pop("embedding"),
    ]
    weights = random_weights(cfg, seed)
    from imparo_amd.config import plan_from_config
    from imparo_amd.engine.model import declared_tensors
    for n, change in enumerate(changes):
        other = copy.deepcopy(cfg)
        change(other)
        d = str(tmp_path / f"other{n}")
        os.makedirs(d)
        with open(os.path.join(d, "config.json"), "w") as fh:
            json.dump(other, fh)
        used = declared_tensors(plan_from_config(other)[1])
        save_file({k: weights[k].to(torch.bfloat16).contiguous() for k in used}, os.path.join(d, "model.safetensors"))
        got = make_engine(d, "float32").step([StepEntry("a", tokens, list(range(60)))]).cpu()
        y = Yardstick(d)
        check(got, y.logits(tokens), f"change {n}", bound("float32", 4), y.noise(tokens))
        assert float((got - base).abs().max()) > 1e-3 * float(base.abs().max()), f"change {n} moves nothing"


def test_generation_through_the_entry_point(models):
    from imparo_amd import generate
    d, y = models["A", "float32"]
    prompts = [prompt_tokens(vocab("A"), n, 50 + n) for n in (1, 6, 29, 13, 40)]
    want = [y.exact.greedy(p, 12) for p in prompts]
    assert all(len(set(w)) > 1 for w in want) and sum(len(set(w)) > 4 for w in want) > 2, f"the plain continuation hardly moves: {want}"
    assert generate(d, prompts, max_tokens=12, dtype="float32", page_size=8) == want
    # three at a time under a small token budget: prompts in portions beside decoding rows
    os.environ["IMPARO_BATCH"] = "5"
    try:
        got = generate(d, prompts, max_tokens=12, dtype="float32", page_size=8, parallel=3, max_batch_tokens=11)
    finally:
        del os.environ["IMPARO_BATCH"]
    assert got == want
    got16 = generate(d, prompts, max_tokens=12, dtype="bfloat16", parallel=3)
    assert all(len(out) == 12 for out in got16)


def test_trace_replay_program(models, tmp_path):
    d, y = models["C", "float32"]
    V = vocab("C")
    tokens, other = prompt_tokens(V, 45, 1), prompt_tokens(V, 9, 2)
    steps = [
        {"step": 0, "entries": [{"id": "a", "tokens": tokens[:20], "want": [0, 19]}], "end": []},
        {"step": 1, "entries": [{"id": "a", "tokens": tokens[20:44], "want": []},
                                {"id": "b", "tokens": other, "want": [8]}], "end": ["b"]},
        {"step": 2, "entries": [{"id": "a", "tokens": tokens[44:], "want": [0]}], "end": ["a"]},
    ]
    out = tmp_path / "out"
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", d, "--dtype", "float32", "--out", str(out),
                        "--max-tokens", "128"], input="\n".join(json.dumps(s) for s in steps) + "\n",
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    assert [l for l in r.stdout.splitlines() if l.startswith("done")] == ["done 0", "done 1", "done 2"]
    ref, ref_other = y.logits(tokens), y.logits(other)
    read = lambda n: torch.from_numpy(np.fromfile(out / f"{n}.f32", dtype="<f4").reshape(-1, V))
    check_logits(read(0), ref[[0, 19]], "float32", "step 0")
    check_logits(read(1), ref_other[[8]], "float32", "step 1")
    check_logits(read(2), ref[[44]], "float32", "step 2")

"""Mixtures whose router rides with the norm before them, served: prompts, captured steps of 1 to 16 rows, steps of 17 and
steps beside a prompt's portion, against the plain implementation and, bit for bit, against the launches one by one."""
import pytest
import torch

import plain_rekezen as plain
from conftest import prompt_tokens
from gpu_helpers import make_engine
from rekezen_models import attention, layer, moe, write_model
from tolerances import bound

pytestmark = pytest.mark.gpu


def config(width, streams):
    heads = dict(softcap=20.0, rot=64, base=1e5, scaling=(4.0, 64, 32.0, 1.0))
    return dict(
        architecture="Rekezen", vocab=150, width=width, norm=dict(eps=1e-5), streams=streams, logit_scale=1.1,
        embedding=dict(bigram=dict(buckets=91, mul_prev=31, mul_cur=5)),
        layers=[
            # a shared unit that is one of the experts; none; one of another size, which keeps the router where it was; a layer
            # without feed-forward behind experts' rows; as many outputs as ride, and one
            layer(attention(4, 2, 64, 64, **heads), moe(64, 1.5, 8, 4, (64, 2.0))),
            layer(attention(4, 2, 64, 64, kv_from=0, **heads), moe(40, 1.5, 5, 3)),
            layer(attention(2, 2, 64, 64, softcap=9.0), moe(32, 2.0, 8, 2, (200, 1.0))),
            layer(attention(2, 1, 128, 128, softcap=9.0), moe(32, 1.0, 16, 8)),
            layer(attention(2, 1, 128, 128, softcap=9.0, kv_from=3), None),
            layer(attention(4, 1, 64, 64, softcap=9.0), moe(96, 1.0, 1, 1)),
        ])


def serve(eng, prompts, fed):
    """Prompts of all but one in one step, then tokens one by one while requests end, the last prompt beside them: logits of
    every token."""
    from imparo_amd.engine import StepEntry
    got = [[] for _ in prompts]

    def step(entries):
        out = eng.step([StepEntry(i, prompts[i][lo:hi], list(range(hi - lo))) for i, lo, hi in entries]).cpu()
        at = 0
        for i, lo, hi in entries:
            got[i].append(out[at:at + hi - lo])
            at += hi - lo

    late = len(prompts) - 1
    step([(i, 0, fed[i]) for i in range(late)])
    done, live = list(fed), list(range(late))
    while live:
        singles = [(i, done[i], done[i] + 1) for i in live]
        joins = len(live) == 8 and not got[late]
        step(singles + [(late, 0, fed[late])] if joins else singles)
        for i in list(live):
            done[i] += 1
            if done[i] == len(prompts[i]):
                eng.release(i)
                live.remove(i)
        if joins:
            live.append(late)
    return [torch.cat(g) for g in got]


@pytest.mark.parametrize("width,streams", [(256, 4), (512, 2), (1024, 3)])
def test_served_with_riding_routers(width, streams, tmp_path, monkeypatch):
    from imparo_amd.kernels import ops
    cfg = config(width, streams)
    d = write_model(cfg, 31, str(tmp_path / "m"), steady=True)
    fed = [1 + 3 * i % 11 for i in range(17)] + [30]
    # (17 rows, 16, 8 and fewer, one: the requests end one after the other)
    prompts = [prompt_tokens(cfg["vocab"], n + 2 + i, 70 + i) for i, n in enumerate(fed)]
    rides, of = [], ops.stream_norm

    def counted(x, *args, route=None, **kw):
        if route is not None:
            rides.append((x.shape[0], route.weight.shape[0]))
        return of(x, *args, route=route, **kw)

    monkeypatch.setattr(ops, "stream_norm", counted)
    got = []
    for riding in (True, False):
        del rides[:]
        eng = make_engine(d, "bfloat16", max_tokens=4096, max_requests=18)
        assert [b.routes for b in eng.model.blocks] == [True, True, True, True, False, True]
        if not riding:
            for b in eng.model.blocks:
                b.routes = False
        got.append(serve(eng, prompts, fed))
        eng.cache.check()
        assert {n for _, n in rides} == ({8, 5, 16, 1} if riding else set())
        if riding:                              # (the third layer's shared unit keeps its router where it was)
            assert {t for t, _ in rides} >= {1, 8, 16} and max(t for t, _ in rides) == 16
            per_step = sum(1 for t, n in rides if t == 8 and n == 8)
            assert sum(1 for t, n in rides if t == 8) == 4 * per_step
    assert all(torch.equal(a, b) for a, b in zip(*got))
    ref, single = plain.PlainRekezen(d), plain.PlainRekezen(d)
    want = [ref.logits(p) for p in prompts]
    scale = max(float(w.abs().max()) for w in want)
    for p, g, w in zip(prompts, got[0], want):
        noise = (single.logits(p, inputs_as=torch.bfloat16) - w).abs().max(dim=-1).values / scale
        allowed = torch.maximum(torch.full_like(noise, bound("bfloat16", len(cfg["layers"]))), 3.0 * noise)
        err = (g.float() - w).abs().max(dim=-1).values / scale
        assert bool((err <= allowed).all()), (float(err.max()), float(allowed.max()))

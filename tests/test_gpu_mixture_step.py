"""A mixture's decode step: the norm that takes the router along, and products that go by the tokens' choices. Both against the
launches they stand for, whose bits they have."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def ops():
    from imparo_amd.kernels import ops
    return ops


def rnd(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


@pytest.mark.parametrize("T,experts,used", [(1, 9, 5), (8, 9, 5), (16, 24, 8), (5, 2, 1), (16, 3, 3)])
@pytest.mark.parametrize("F,E", [(32, 8), (768, 1024), (96, 200), (160, 2056)])
def test_products_by_the_tokens_choices_have_the_planned_bits(T, experts, used, F, E):
    choice = torch.stack([torch.randperm(experts + 1, generator=torch.Generator().manual_seed(i))[:used] for i in range(T)])
    choice[choice == experts] = experts + 7                      # (an expert past the last one: nobody's entry)
    choice = choice.to(torch.int32).to(DEV)
    n, up, down = rnd(T, E, seed=1, dtype=torch.bfloat16), rnd(experts, 2 * F, E, seed=2, dtype=torch.bfloat16), rnd(experts, E, F, seed=3, dtype=torch.bfloat16)
    limits = torch.linspace(0.5, 9.0, experts, device=DEV)
    limits[0] = 0.0
    entries = T * used
    rows = 16
    tiles = torch.empty(ops().moe_max_tiles(entries, experts, rows), 3, dtype=torch.int32, device=DEV)
    slot, entry = (torch.zeros(entries, dtype=torch.int32, device=DEV) for _ in range(2))
    ops().moe_plan(choice, experts, rows, slot, entry, tiles)
    hidden, y = torch.zeros(entries, F, dtype=torch.bfloat16, device=DEV), torch.zeros(entries, E, device=DEV)
    ops().moe_gemm(n, up, hidden, tiles, rows, entry, gather_div=used, epilogue="gated", limits=limits, alpha=1.702)
    ops().moe_gemm(hidden, down, y, tiles, rows)
    hidden_d, y_d = torch.full((entries, F), 3.0, dtype=torch.bfloat16, device=DEV), torch.full((entries, E), 7.0, device=DEV)
    ops().moe_gemm_direct(n, up, hidden_d, choice, own_rows=True, epilogue="gated", limits=limits, alpha=1.702)
    ops().moe_gemm_direct(hidden_d, down, y_d, choice)
    has = slot >= 0
    at = slot[has].long()
    assert torch.equal(hidden_d[has], hidden[at]) and torch.equal(y_d[has], y[at])
    assert bool((hidden_d[~has] == 3.0).all()) and bool((y_d[~has] == 7.0).all())


@pytest.mark.parametrize("T,width,streams,in_streams", [(1, 256, 1, 1), (8, 1024, 4, 4), (16, 2048, 3, 1), (3, 768, 2, 2), (5, 4096, 4, 4)])
@pytest.mark.parametrize("pending", ["one", "slices", "experts"])
@pytest.mark.parametrize("norm", ["rms", "layer", "none"])
def test_the_step_norm_and_its_router_have_the_bits_of_their_launches(T, width, streams, in_streams, pending, norm, monkeypatch):
    x = rnd(T, in_streams, width, seed=1) if in_streams > 1 else rnd(T, width, seed=1)
    weight, bias = rnd(width, seed=2), (None if norm == "rms" else rnd(width, seed=3))
    mix, join, read = rnd(streams, streams, seed=4), rnd(streams, seed=5), rnd(streams, seed=6)
    if pending == "experts":
        choice = torch.stack([torch.randperm(11, generator=torch.Generator().manual_seed(i))[:6] for i in range(T)]).to(torch.int32).to(DEV)
        delta = types.SimpleNamespace(y=rnd(T * 6, width, seed=7), h=rnd(T, width, seed=8, dtype=torch.bfloat16), choice=choice,
                                      weight=rnd(T, 6, seed=9).abs(), slot_of_entry=torch.arange(T * 6, dtype=torch.int32, device=DEV),
                                      n_experts=9, extra=None, by_entry=True)     # (experts 9 and 10 hand their input on)
    else:
        delta = rnd(T, width, seed=7) if pending == "one" else rnd(3, T, width, seed=7)
    router, top, always = rnd(8, width, seed=10, dtype=torch.bfloat16), 4, 1
    correction = rnd(8, seed=11)
    got = []
    for step in (True, False):
        out, moved = torch.empty(T, width, dtype=torch.bfloat16, device=DEV), torch.empty(T, streams, width, device=DEV)
        chosen, shares = torch.empty(T, top + always, dtype=torch.int32, device=DEV), torch.empty(T, top + always, device=DEV)
        call = dict(delta=delta, mix=mix, join=join, read=read, x_out=moved)
        rides = ops().stream_step_routes(x, delta, streams, weight, bias, router, top)
        assert rides == (step and width in (256, 768, 1024, 2048))
        if rides:
            ride = types.SimpleNamespace(weight=router, bias=None, correction=correction, top=top, always=always, scoring="chosen",
                                         normalize=False, scale=1.25, choice=chosen, shares=shares)
            ops().stream_norm(x, norm, weight, bias, 1e-5, out, route=ride, **call)
        else:
            ops().stream_norm(x, norm, weight, bias, 1e-5, out, **call)
            z = torch.empty(T, 8, device=DEV)
            ops().gemm(out, router, z)
            ops().moe_route(z, correction, chosen, shares, top, scoring="chosen", n_router=8, groups=1, keep=1, normalize=False, scale=1.25,
                            always=always)
        got.append((out, moved, chosen, shares))
        monkeypatch.setattr(ops(), "_stream_step_takes", lambda *a: False)
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("before,always,taken", [(5, 1, True), (6, 1, False), (4, 1, False)])
def test_choices_in_place_of_the_ones_that_join(before, always, taken):
    """A router that rides behind experts' rows may write its choices where theirs lay if the rows are as long; of other lengths a
    row's choices would lie where another row's are still read, and the call is refused."""
    from imparo_amd.kernels import KernelArgumentError
    T, width, top = 16, 1024, 4
    used = top + always
    x, weight, router = rnd(T, width, seed=1), rnd(width, seed=2), rnd(8, width, seed=3, dtype=torch.bfloat16)
    choice = torch.stack([torch.randperm(9, generator=torch.Generator().manual_seed(i))[:before] for i in range(T)]).to(torch.int32).to(DEV)
    shares = rnd(T, before, seed=4).abs()
    y, h = rnd(T * before, width, seed=5), rnd(T, width, seed=6, dtype=torch.bfloat16)
    got = []
    for shared in (False, True):
        buffers = [torch.zeros(T * 8, dtype=t.dtype, device=DEV) for t in (choice, shares)]
        joins = [b[:T * before].view(T, before).copy_(t) for b, t in zip(buffers, (choice, shares))]
        chosen = [b[:T * used].view(T, used) if shared else torch.zeros(T, used, dtype=b.dtype, device=DEV) for b in buffers]
        delta = types.SimpleNamespace(y=y, h=h, choice=joins[0], weight=joins[1], n_experts=9, extra=None, by_entry=True,
                                      slot_of_entry=torch.arange(T * before, dtype=torch.int32, device=DEV))
        ride = types.SimpleNamespace(weight=router, bias=None, correction=None, top=top, always=always, scoring="chosen", normalize=False,
                                     scale=1.0, choice=chosen[0], shares=chosen[1])
        out, moved = torch.empty(T, width, dtype=torch.bfloat16, device=DEV), torch.empty(T, 1, width, device=DEV)
        run = lambda: ops().stream_norm(x, "rms", weight, None, 1e-5, out, delta=delta, x_out=moved, streams=1, route=ride)
        if shared and not taken:
            with pytest.raises(KernelArgumentError):
                run()
            return
        run()
        got.append((out, moved, *chosen))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("width", [256, 512, 768, 1024, 2048])
@pytest.mark.parametrize("outputs,top,always", [(1, 1, 0), (5, 3, 1), (8, 4, 1), (9, 1, 2), (16, 8, 0), (16, 16, 3)])
@pytest.mark.parametrize("biased,corrected", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("scoring,normalize", [("chosen", False), ("softmax", True), ("sigmoid", False)])
def test_riding_routers_of_all_forms(width, outputs, top, always, biased, corrected, scoring, normalize):
    """Choices and weights as the norm, the product of few rows with its bias, and the choice leave them in launches of their own."""
    T, streams = 7, 3
    x, delta = rnd(T, streams, width, seed=1), rnd(T, width, seed=2)
    weight, bias = rnd(width, seed=3), rnd(width, seed=4)
    mix, join, read = rnd(streams, streams, seed=5), rnd(streams, seed=6), rnd(streams, seed=7)
    router = (rnd(outputs, width, seed=8) * width ** -0.5).to(torch.bfloat16)
    router_bias, correction = rnd(outputs, seed=9) if biased else None, 0.3 * rnd(outputs, seed=10) if corrected else None
    used = top + always
    assert ops().stream_step_routes(x, delta, streams, weight, bias, router, top)
    got = []
    for rides in (True, False):
        out, moved = torch.empty(T, width, dtype=torch.bfloat16, device=DEV), torch.empty(T, streams, width, device=DEV)
        chosen, shares = torch.full((T, used), -7, dtype=torch.int32, device=DEV), torch.full((T, used), -7.0, device=DEV)
        call = dict(delta=delta, mix=mix, join=join, read=read, x_out=moved)
        if rides:
            ride = types.SimpleNamespace(weight=router, bias=router_bias, correction=correction, top=top, always=always, scoring=scoring,
                                         normalize=normalize, scale=1.25, choice=chosen, shares=shares)
            ops().stream_norm(x, "layer", weight, bias, 1e-5, out, route=ride, **call)
        else:
            ops().stream_norm(x, "layer", weight, bias, 1e-5, out, **call)
            z = torch.empty(T, outputs, device=DEV)
            ops().gemm(out, router, z, bias=router_bias)
            ops().moe_route(z, correction, chosen, shares, top, scoring=scoring, normalize=normalize, scale=1.25, always=always)
        got.append((out, moved, chosen, shares))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    z = got[0][0].double() @ router.double().t() + (0 if router_bias is None else router_bias.double())
    score = {"chosen": z, "softmax": torch.softmax(z, -1), "sigmoid": torch.sigmoid(z)}[scoring]
    ranked = (score if correction is None else score + correction.double()).sort(-1, descending=True)
    # (where no rounding of a sum of products of about one turns a choice)
    sure = ((ranked.values[:, :-1] - ranked.values[:, 1:])[:, :top] > 1e-5).all(-1) if outputs > 1 else torch.ones(T, dtype=torch.bool, device=DEV)
    assert torch.equal(got[0][2][sure, :top].long(), ranked.indices[sure, :top])
    assert torch.equal(got[0][2][:, top:].cpu(), (outputs + torch.arange(always, dtype=torch.int32)).expand(T, always))

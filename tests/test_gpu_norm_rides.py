"""A norm without a statistic in the launch of the product before it: against the two launches, and whole models with and without."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


# one block partly past the end, more columns than blocks of 8, one chunk of K, a ragged K, two chains of sums
@pytest.mark.parametrize("n, k", [(8, 128), (41, 72), (1024, 1024), (130, 3072), (72, 4096), (2056, 4224)])
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("biased", [False, True])
def test_product_with_the_norm_behind_it(n, k, m, biased):
    x, w = rnd(m, k, seed=1).bfloat16().to(DEV), rnd(n, k, seed=2, scale=0.05).bfloat16().to(DEV)
    b = rnd(n, seed=3).to(DEV) if biased else None
    held, nw, nb = (rnd(*s, seed=i).to(DEV) for i, s in ((4, (m, n)), (5, (n,)), (6, (n,))))
    stream = held.clone()
    rows = torch.full((m, n), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.rows_gemm_tanh(x, w, stream, bias=b, out=rows, alpha=0.7, norm_weight=nw, norm_bias=nb)
    y = x.double() @ w.double().t() + (0.0 if b is None else b.double())
    # a float32 sum of k products and of two more terms, in any order
    bound = (x.double().abs() @ w.double().abs().t() + held.double().abs() + 4.0) * (k + 3) * 2.0 ** -24
    assert bool(((stream.double() - (held.double() + y)).abs() <= bound).all())
    want = torch.empty_like(rows)
    ops.dynamic_tanh(stream, 0.7, nw, nb, want, ())
    assert torch.equal(rows, want)                           # the rows that the norm's own launch makes of that stream
    alone = held.clone()
    ops.rows_gemm_tanh(x, w, alone, bias=b)
    assert torch.equal(alone, stream)
    # and no further from 64 bits than the slices of K that it stands for, added in order
    slices = ops.gemm_slices(m, n, k, torch.bfloat16)
    if slices > 1 and k <= 4096 and not biased:
        parts, zero = torch.empty(slices, m, n, device=DEV), torch.zeros(m, n, device=DEV)
        ops.gemm(x, w, parts)
        ops.rows_gemm_tanh(x, w, zero)
        total = parts[0]
        for part in parts[1:]:
            total = total + part
        # (errors of 8e-8 over thousands of outputs; a tenth is more than samples of one row differ by)
        assert float((zero.double() - y).norm()) <= 1.1 * float((total.double() - y).norm())
    with pytest.raises(ops.KernelArgumentError):
        ops.rows_gemm_tanh(x, w, alone, out=rows, alpha=0.7)
    with pytest.raises(ops.KernelArgumentError):
        ops.rows_gemm_tanh(x, w, alone[:, :n - 1].contiguous())


# weights that ride and that do not, at the lines between them
@pytest.mark.parametrize("n, k, rides", [(1024, 3072, True), (1024, 3080, False), (1032, 4096, True), (2048, 4104, False), (2056, 2048, True),
                                         (2056, 2056, False), (4104, 1024, True), (4104, 1032, False), (6152, 512, True), (8200, 256, False)])
def test_a_row_is_summed_in_one_order_in_all_steps_of_few_rows(n, k, rides):
    """A request's stream and rows do not depend on how many others decode beside it."""
    import types
    from imparo_amd.parts.base import NormRide, Residual, Workspace
    from imparo_amd.parts.linear import Linear
    from imparo_amd.parts.norm import DynamicTanh
    x, held = rnd(16, k, seed=1).bfloat16().to(DEV), rnd(16, n, seed=2).to(DEV)
    linear = Linear(rnd(n, k, seed=3, scale=k ** -0.5).bfloat16().to(DEV))
    norm = DynamicTanh.__new__(DynamicTanh)
    norm.alpha, norm.weight, norm.bias = 0.7, rnd(n, seed=4).to(DEV), rnd(n, seed=5).to(DEV)
    first = None
    for m in (16, 1, 2, 4, 8, 9, 12, 13, 15):
        res = Residual(held[:m].clone())
        ctx = types.SimpleNamespace(workspace=Workspace(torch.device(DEV)), stream=res.x, ride=NormRide(norm, torch.bfloat16))
        delta = linear(ctx, x[:m], torch.float32, "out", sliced_ok=True, into=res.x)
        assert (ctx.ride.rows is not None) == rides and (delta is res.x) == rides
        res.pending, res.normed = (None, ctx.ride) if rides else (delta, None)
        rows = norm.forward(ctx, res, torch.bfloat16)
        first = first if first is not None else (res.x.clone(), rows.clone())
        assert torch.equal(res.x, first[0][:m]) and torch.equal(rows, first[1][:m])


def test_a_models_steps_with_and_without(tmp_path, monkeypatch):
    """Prompts and decoded tokens of a model whose layers' norms ride (delta rule, and attention beside lightning attention)."""
    from imparo_amd import Engine, StepEntry, write_random_model
    from imparo_amd.parts import linear
    mixers = [dict(type="channel_delta", mixer=dict(heads=2, kv_heads=1, dim=128, vdim=128, conv=4)),
              dict(type="parallel", mixer=dict(
                  left=dict(heads=4, kv_heads=2, dim=64, vdim=64, scale=0.125, softcap=30.0, mask=dict(size=64, keep_first=4),
                            rot=dict(dims=64, base=10000.0)),
                  right=dict(heads=2, dim=128, vdim=128, decay=[0.9, 0.99]), left_scale=0.8, right_scale=0.6))]
    config = dict(architecture="Vebusun", vocab=256, width=256, norm=dict(eps=1e-5), residual_mult=0.5, embedding=dict(scale=1.0),
                  layers=[dict(mixers[i % 2], mlp=dict(kind="dense", ff=512)) for i in range(4)])
    folder = str(tmp_path)
    write_random_model(config, 3, folder, layer_gain=4.0)
    calls, ride = [], ops.rows_gemm_tanh
    monkeypatch.setattr(ops, "rows_gemm_tanh", lambda *a, **k: (calls.append(k.get("out") is not None), ride(*a, **k))[1])
    results = []
    for most in (linear.RIDE_MAX_K, 0):
        monkeypatch.setattr(linear, "RIDE_MAX_K", most)
        engine, logits = Engine(folder, dtype="bfloat16", max_tokens=512, max_requests=4), []
        for step in range(5):
            tokens = [[(7 * i + j) % 256 for j in range(5 + i)] if step == 0 else [(31 * step + i) % 256] for i in range(3)]
            logits.append(engine.step([StepEntry(i, t, [len(t) - 1]) for i, t in enumerate(tokens)]).clone())
        results.append((torch.stack(logits), len(calls), sum(calls)))
        calls.clear()
    # the first step's 18 tokens have kernels of their own; then every product into the stream but a last block's way back rides
    (with_, n, normed), (without, none, _) = results
    assert n > 0 and n % 9 == 0 and normed * 9 == n * 7 and none == 0
    # (bfloat16 rows of the same float32 stream, whose sums come in another order)
    assert float((with_ - without).norm() / without.norm()) < 0.02

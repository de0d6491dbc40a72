"""A decode step of the channel delta rule in one launch against the launches it stands for."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("heads, kv_heads", [(1, 1), (2, 1), (3, 3), (8, 4)])
@pytest.mark.parametrize("taps", [1, 2, 4])
@pytest.mark.parametrize("rows_n", [1, 5])
def test_one_launch_is_the_four(heads, kv_heads, taps, rows_n):
    g = torch.Generator().manual_seed(heads * 100 + taps * 10 + rows_n)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(DEV)
    D, H, Hk, slots = 128, heads, kv_heads, rows_n + 3
    C = (2 * Hk + H) * D
    rows, steps = rnd(rows_n, C + H + 8), rnd(rows_n, 2 * H * D)
    conv_w, conv = rnd(C, taps, scale=0.5), rnd(slots, taps - 1, C)
    bias, rate = rnd(H * D, scale=0.5), rnd(H).exp() * 0.1
    state, norm = rnd(slots, H, D, D, scale=0.3), rnd(H * D)
    slot = torch.randperm(slots, generator=g)[:rows_n].int().to(DEV)
    single = torch.arange(rows_n, device=DEV, dtype=torch.int32)
    ones = torch.ones(rows_n, device=DEV, dtype=torch.int32)
    state2, conv2 = state.clone(), conv.clone()
    qkv, o = torch.empty(rows_n, C, device=DEV), torch.empty(rows_n, H * D, device=DEV)
    ops.causal_conv(rows, C, conv_w, None, conv2 if taps > 1 else None, single, single, ones, slot, qkv, silu=True, single_tokens=True)
    ops.head_prepare(qkv, 0, 2 * Hk, D, unit=True, unit_eps=1e-6, n_first=Hk, scale_first=D ** -0.5)
    ops.channel_delta_scan(qkv, 0, H // Hk, qkv, Hk * D, H // Hk, qkv, 2 * Hk * D, steps, 0, bias, rate, rows, C, state2, single, ones,
                           slot, o, H, D, D)
    want = torch.empty(rows_n, H * D, device=DEV)
    ops.gated_group_norm(o, steps, H * D, norm, H, 1e-5, want, gate_first=False, gate_act="sigmoid")
    got = torch.full_like(want, float("nan"))
    ops.channel_delta_step(rows, C, steps, H * D, conv_w, conv if taps > 1 else None, bias, rate, state, slot, norm, got, H, Hk, D, D,
                           1e-6, D ** -0.5, 1e-5)
    # sums of 128 products in another order, 128 roundings of 6e-8 at the most, over values of order one
    assert torch.equal(conv, conv2)
    torch.testing.assert_close(state, state2, rtol=2e-5, atol=2e-5)
    torch.testing.assert_close(got, want, rtol=2e-4, atol=2e-4)
    half = torch.empty(rows_n, H * D, device=DEV, dtype=torch.bfloat16)
    assert not ops.channel_delta_step_takes(H, Hk, 64, 128, taps) and not ops.channel_delta_step_takes(3 * Hk, Hk, D, D, taps)
    with pytest.raises(ops.KernelArgumentError):
        ops.channel_delta_step(rows[:, :C].contiguous(), C, steps, H * D, conv_w, conv, bias, rate, state, slot, norm, half, H, Hk, D, D,
                               1e-6, 1.0, 1e-5)


@pytest.mark.parametrize("heads, kv_heads, taps", [(1, 1, 4), (4, 2, 3)])
def test_bfloat16_out_is_the_float32_rounded(heads, kv_heads, taps):
    """What a bfloat16 engine reads, and a second step on what the first one left."""
    g = torch.Generator().manual_seed(heads)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(DEV)
    D, H, Hk, n, slots = 128, heads, kv_heads, 3, 4
    C = (2 * Hk + H) * D
    conv_w, conv, state = rnd(C, taps, scale=0.5), rnd(slots, taps - 1, C), rnd(slots, H, D, D, scale=0.3)
    bias, rate, norm = rnd(H * D, scale=0.5), rnd(H).exp() * 0.1, rnd(H * D)
    slot = torch.tensor([2, 0, 3], device=DEV, dtype=torch.int32)
    sides = [(conv.clone(), state.clone(), torch.full((n, H * D), float("nan"), device=DEV, dtype=t)) for t in (torch.float32, torch.bfloat16)]
    for _ in range(2):
        rows, steps = rnd(n, C + H), rnd(n, 2 * H * D)
        for history, kept, out in sides:
            ops.channel_delta_step(rows, C, steps, H * D, conv_w, history, bias, rate, kept, slot, norm, out, H, Hk, D, D, 1e-6,
                                   D ** -0.5, 1e-5)
        (history, kept, whole), (history2, kept2, half) = sides
        assert torch.equal(half, whole.bfloat16()) and torch.equal(history, history2) and torch.equal(kept, kept2)
    assert torch.equal(kept[1], state[1]) and torch.equal(history[1], conv[1])       # nobody's slot

"""The projection with the conv in its launch, and a head a block behind it, against the launches they stand for."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one tile and a part of one, the conv's last channel inside a tile, no other column, one tile of two a block; one chunk of K, more
# than the waves, a ragged one
@pytest.mark.parametrize("n, channels, k", [(20, 12, 128), (384, 384, 256), (2312, 2048, 1024), (531, 512, 1160), (5000, 4096, 3072)])
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("taps", [1, 2, 4])
def test_projection_with_the_conv(n, channels, k, m, taps):
    g = torch.Generator().manual_seed(n + m)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(DEV)
    x, w = rnd(m, k).bfloat16(), rnd(n, k, scale=k ** -0.5).bfloat16()
    slots = m + 2
    conv_w, conv = rnd(channels, taps, scale=0.5), rnd(slots, taps - 1, channels)
    slot = torch.randperm(slots, generator=g)[:m].int().to(DEV)
    conv2, plain = conv.clone(), torch.empty(m, n, device=DEV)
    ops.gemm(x, w, plain)
    single, ones = torch.arange(m, device=DEV, dtype=torch.int32), torch.ones(m, device=DEV, dtype=torch.int32)
    want = torch.empty(m, channels, device=DEV)
    ops.causal_conv(plain, channels, conv_w, None, conv2 if taps > 1 else None, single, single, ones, slot, want, silu=True,
                    single_tokens=True)
    got = torch.full((m, n), float("nan"), device=DEV)
    ops.rows_gemm_conv(x, w, conv_w, conv if taps > 1 else None, slot, got)
    # sums of k products of unit size in another order, then a few operations
    torch.testing.assert_close(got[:, :channels], want, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(got[:, channels:], plain[:, channels:], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(conv, conv2, rtol=1e-5, atol=1e-5)
    others = [s for s in range(slots) if s not in slot.tolist()]
    assert torch.equal(conv[others], conv2[others])
    with pytest.raises(ops.KernelArgumentError):
        ops.rows_gemm_conv(x, w, conv_w[:channels - 2].contiguous(), conv, slot, got)


@pytest.mark.parametrize("heads, kv_heads, ranks", [(1, 1, (8, 128)), (2, 1, (128, 128)), (6, 2, (40, 24)), (8, 4, (128, 64))])
@pytest.mark.parametrize("rows_n", [1, 5, 16])
def test_a_head_a_block_is_the_step(heads, kv_heads, ranks, rows_n):
    g = torch.Generator().manual_seed(heads * 100 + rows_n)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(DEV)
    D, H, Hk, slots = 128, heads, kv_heads, rows_n + 3
    C, (ra, rg) = (2 * Hk + H) * D, ranks
    rows = rnd(rows_n, C + H + ra + rg + 3)
    high = rnd(2 * H * D, ra + rg + 8, scale=0.1).bfloat16()
    high[:H * D, ra:] = 0
    high[H * D:, :ra] = 0
    high[H * D:, ra + rg:] = 0
    bias, rate = rnd(H * D, scale=0.5), rnd(H).exp() * 0.1
    state, norm = rnd(slots, H, D, D, scale=0.3), rnd(H * D)
    slot = torch.randperm(slots, generator=g)[:rows_n].int().to(DEV)
    low = torch.zeros(rows_n, ra + rg + 8, device=DEV, dtype=torch.bfloat16)
    low[:, :ra + rg] = rows[:, C + H:C + H + ra + rg].bfloat16()
    steps = (low.double() @ high.double().t()).float()
    single, ones = torch.arange(rows_n, device=DEV, dtype=torch.int32), torch.ones(rows_n, device=DEV, dtype=torch.int32)
    state2, qkv, o = state.clone(), rows[:, :C].contiguous(), torch.empty(rows_n, H * D, device=DEV)
    ops.head_prepare(qkv, 0, 2 * Hk, D, unit=True, unit_eps=1e-6, n_first=Hk, scale_first=D ** -0.5)
    ops.channel_delta_scan(qkv, 0, H // Hk, qkv, Hk * D, H // Hk, qkv, 2 * Hk * D, steps, 0, bias, rate, rows, C, state2, single, ones,
                           slot, o, H, D, D)
    want = torch.empty(rows_n, H * D, device=DEV)
    ops.gated_group_norm(o, steps, H * D, norm, H, 1e-5, want, gate_first=False, gate_act="sigmoid")
    got, half, state3 = torch.full_like(want, float("nan")), torch.empty_like(want, dtype=torch.bfloat16), state.clone()
    for out, kept in ((got, state), (half, state3)):
        ops.channel_delta_heads(rows, C, C + H, high, ra, rg, bias, rate, kept, slot, norm, out, H, Hk, 1e-6, D ** -0.5, 1e-5)
    # sums of 128 products in another order, 128 roundings of 6e-8 at the most, over values of order one
    torch.testing.assert_close(state, state2, rtol=2e-5, atol=2e-5)
    torch.testing.assert_close(got, want, rtol=2e-4, atol=2e-4)
    assert torch.equal(half, got.bfloat16()) and torch.equal(state3, state)
    others = [s for s in range(slots) if s not in slot.tolist()]
    assert torch.equal(state[others], state2[others])
    assert not ops.channel_delta_heads_takes(H, Hk, D, D, 4, 136, 8) and not ops.channel_delta_heads_takes(H, Hk, 64, D, 4, 8, 8)
    with pytest.raises(ops.KernelArgumentError):
        ops.channel_delta_heads(rows[:, :C + H].contiguous(), C, C + H, high, ra, rg, bias, rate, state, slot, norm, got, H, Hk, 1e-6,
                                1.0, 1e-5)

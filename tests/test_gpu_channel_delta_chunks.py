"""The delta rule with decays a channel in chunks, around the ends of chunks, against the recurrence in 64 bits."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("strength", [0.3, 20.0])        # a chunk keeps half of the state; a token hardly anything
@pytest.mark.parametrize("d, dv", [(64, 16), (65, 17), (128, 128)])
def test_chunks_are_the_recurrence(d, dv, strength):
    H, Hk, lens = 4, 2, [64, 65, 95, 96, 97, 3, 129]
    g = torch.Generator().manual_seed(d)
    n, C = sum(lens), 2 * Hk * d + H * dv
    rows = torch.randn(n, C + H, generator=g)                            # q | k | v | b
    heads = rows[:, :2 * Hk * d].view(n, 2 * Hk, d)
    heads /= heads.norm(dim=-1, keepdim=True)
    steps, bias = torch.randn(n, H * d, generator=g), torch.randn(H * d, generator=g) - 1.0
    rate, state = strength * (torch.rand(H, generator=g) + 0.1), torch.randn(len(lens), H, d, dv, generator=g)
    starts = [sum(lens[:i]) for i in range(len(lens))]
    out, S = torch.full((n, H * dv), float("nan"), device=DEV), state.to(DEV)
    chunk_tokens, max_chunks = ops.channel_delta_chunks(max(lens), d)
    assert chunk_tokens == 32
    scratch = torch.full((ops.channel_delta_scratch(len(lens), max_chunks, H, d),), float("nan"), device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    x = rows.to(DEV)
    ops.channel_delta_scan(x, 0, H // Hk, x, Hk * d, H // Hk, x, 2 * Hk * d, steps.to(DEV), 0, bias.to(DEV), rate.to(DEV), x, C, S,
                           i32(starts), i32(lens), i32(list(range(len(lens)))), out, H, d, dv, chunk_tokens=chunk_tokens,
                           max_chunks=max_chunks, scratch=scratch)
    rows, steps, bias, rate, state = (t.double() for t in (rows, steps, bias, rate, state))
    decay = torch.exp(-rate[:, None] * torch.nn.functional.softplus(steps + bias).view(n, H, d))
    want = torch.empty(n, H, dv, dtype=torch.float64)
    q, k = (rows[:, a * Hk * d:(a + 1) * Hk * d].view(n, Hk, d).repeat_interleave(H // Hk, 1) for a in (0, 1))
    v, beta = rows[:, 2 * Hk * d:C].view(n, H, dv), torch.sigmoid(rows[:, C:])
    for r, (first, length) in enumerate(zip(starts, lens)):
        Z = state[r]
        for t in range(first, first + length):
            Z = decay[t][:, :, None] * Z
            Z = Z + k[t][:, :, None] * (beta[t][:, None] * (v[t] - (Z * k[t][:, :, None]).sum(1)))[:, None, :]
            want[t] = (Z * q[t][:, :, None]).sum(1)
        state[r] = Z
    # sums of up to 128 products and of a triangle's 32, four roundings a term, and of 20 steps' logarithms in a decay: some 2,000
    # roundings of 6e-8, which add up as their root
    error = lambda got, ref: ((got.cpu().double() - ref).norm() / ref.norm()).item()
    assert error(out, want.view(n, -1)) < 5e-6
    assert error(S, state) < 5e-6


@pytest.mark.parametrize("d", [4, 33, 64, 65, 128])
def test_a_pairs_sum_runs_over_the_state_rows_in_order(d):
    # nothing decays and the first token alone has a key, of ones, and values of one: the result of token t in its chunk is then the sum of
    # its query, one number after the other in float32, and everything else on the way is exact
    H, dv, n = 2, 16, 64
    q = torch.randn(n, H, d, generator=torch.Generator().manual_seed(d)) * 2.0 ** torch.arange(n)[:, None, None].remainder(5)
    k, v = torch.zeros(n, H, d), torch.zeros(n, H, dv)
    k[0], v[0] = 1.0, 1.0
    rows = torch.cat([q.reshape(n, -1), k.view(n, -1), v.view(n, -1), torch.full((n, H), 100.0)], 1).to(DEV)
    out, S = torch.empty(n, H * dv, device=DEV), torch.zeros(1, H, d, dv, device=DEV)
    chunk_tokens, max_chunks = ops.channel_delta_chunks(n, d)
    scratch = torch.empty(ops.channel_delta_scratch(1, max_chunks, H, d), device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ops.channel_delta_scan(rows, 0, 1, rows, H * d, 1, rows, 2 * H * d, torch.zeros(n, H * d, device=DEV), 0, torch.zeros(H * d, device=DEV),
                           torch.zeros(H, device=DEV), rows, 2 * H * d + H * dv, S, i32([0]), i32([n]), i32([0]), out, H, d, dv,
                           chunk_tokens=chunk_tokens, max_chunks=max_chunks, scratch=scratch)
    want = torch.zeros(n, H)
    for i in range(d):
        want += q[:, :, i]
    assert torch.equal(out.cpu().view(n, H, dv)[:chunk_tokens], want[:chunk_tokens, :, None].expand(-1, -1, dv))

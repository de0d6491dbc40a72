"""A prompt's router, choice and plan in two launches, against 64 bits and bit for bit against the launches for each."""
import pytest
import torch

from imparo_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# outputs up to the 32 of a product; K of one step of 128 up to more than the 1,024 that lie in LDS at once; tokens around blocks
# of 16 and of 64; with outputs that stand for no expert, and with experts that every token uses
@pytest.mark.parametrize("n_router, n_experts, top, always, k, scoring", [
    (8, 9, 4, 1, 1024, "chosen"), (1, 1, 1, 0, 128, "softmax"), (16, 14, 3, 0, 256, "sigmoid"), (17, 17, 2, 0, 1152, "softmax"),
    (32, 32, 16, 0, 2048, "chosen"), (28, 32, 4, 4, 2944, "softmax")])
@pytest.mark.parametrize("T", [129, 192, 333, 2081])
def test_router_plan(n_router, n_experts, top, always, k, scoring, T):
    assert ops.moe_router_takes(T, n_router, n_experts, top, 1, always, k)
    assert not ops.moe_router_takes(128, n_router, n_experts, top, 1, always, k)
    g = torch.Generator().manual_seed(T * 100 + n_router)
    x, w = torch.randn(T, k, generator=g).bfloat16(), (torch.randn(n_router, k, generator=g) / k ** 0.5).bfloat16()
    bias, correction = torch.randn(n_router, generator=g), 0.1 * torch.randn(n_router, generator=g)
    used, entries = top + always, T * (top + always)
    i32 = lambda *shape: torch.full(shape, -77, dtype=torch.int32, device=DEV)
    choice, weight, counts = i32(T, used), torch.empty(T, used, device=DEV), i32(ops.moe_router_blocks(T), n_experts)
    rows = 64
    slot, entry, tiles = i32(entries), i32(entries), i32(ops.moe_max_tiles(entries, n_experts, rows), 3)
    dev = lambda t: t.to(DEV)
    ops.moe_router_plan(dev(x), dev(w), dev(bias), dev(correction), choice, weight, counts, top, n_experts, rows, slot, entry, tiles,
                        scoring=scoring, normalize=True, scale=1.5, always=always)
    # the same bits as by the product and the choice in launches of their own
    logits, choice_too, weight_too = torch.empty(T, n_router, device=DEV), torch.empty_like(choice), torch.empty_like(weight)
    ops.gemm(dev(x), dev(w), logits, bias=dev(bias))
    ops.moe_route(logits, dev(correction), choice_too, weight_too, top, scoring=scoring, normalize=True, scale=1.5, always=always)
    assert torch.equal(choice, choice_too) and torch.equal(weight, weight_too)
    # the choice that 64 bits make, where no rounding of a sum of k products (2^-24 a product of logits of about one) turns it
    z = x.double() @ w.double().t() + bias.double()
    score = {"chosen": z, "sigmoid": torch.sigmoid(z), "softmax": torch.softmax(z, -1)}[scoring]
    ranked, order = torch.sort(score + correction.double(), descending=True, dim=-1)
    gaps = ranked[:, :-1] - ranked[:, 1:]
    sure = (gaps[:, :top] > 1e-5).all(-1) if n_router > 1 else torch.ones(T, dtype=torch.bool)
    assert sure.float().mean() > 0.9
    got = choice.cpu()
    assert torch.equal(got[sure, :top].long(), order[sure, :top])
    assert torch.equal(got[:, top:], (n_router + torch.arange(always)).expand(T, always).to(torch.int32))
    want = torch.gather(score, 1, order[:, :top])
    want = torch.softmax(want, -1) * 1.5 if scoring == "chosen" else want / want.sum(-1, keepdim=True) * 1.5
    # (2^-24 times the root of k products, the exponential's and the division's own roundings, of weights up to 1.5)
    torch.testing.assert_close(weight.cpu()[sure, :top].double(), want[sure], rtol=2e-5, atol=2e-6)
    assert (weight[:, top:] == 1).all()
    # the plan of these choices: the same tiles, and every entry of an expert in a slot of its own among the expert's
    slot_too, entry_too, tiles_too = torch.empty_like(slot), torch.empty_like(entry), torch.empty_like(tiles)
    ops.moe_plan(choice, n_experts, rows, slot_too, entry_too, tiles_too)
    assert torch.equal(tiles, tiles_too)
    e, s = got.flatten().long(), slot.cpu().long()
    real = e < n_experts
    assert (s[~real] == -1).all()
    assert torch.equal(torch.sort(s[real]).values, torch.arange(int(real.sum())))
    assert torch.equal(entry.cpu().long()[s[real]], torch.nonzero(real).flatten())
    of_slot = torch.empty(int(real.sum()), dtype=torch.long)
    of_slot[s[real]] = e[real]
    assert (of_slot[1:] >= of_slot[:-1]).all()

"""Which norms ride with the product before them: those whose `ride` describes the `forward` they run, behind a part whose
`forward` ends with its product into the stream. Who replaces one `forward` alone gets the launches one by one."""
import types

import pytest
import torch

from imparo_amd.parts import attention, channel_delta, ffn, mixer_pair, moe, norm, retention
from imparo_amd.parts.base import Residual, emits
from imparo_amd.parts.block import HyperBlock, PreNormBlock


new = lambda cls: cls.__new__(cls)


@pytest.mark.parametrize("part", [ffn.SwiGlu, ffn.ClampedGlu, ffn.PolyNormFfn, attention.Attention, channel_delta.ChannelDelta,
                                  retention.Retention, mixer_pair.MixerPair])
def test_parts_that_end_with_their_product_say_so(part):
    class Further(part):
        def forward(self, *args):
            raise NotImplementedError

    block = PreNormBlock(dict(mixer_norm=new(norm.DynamicTanh), mixer=new(part), ffn_norm=new(norm.DynamicTanh), ffn=new(part)))
    assert block.mixer_takes and block.ffn_takes and block.first_rides and block.ffn_norm_rides
    block = PreNormBlock(dict(mixer_norm=new(norm.RmsNorm), mixer=new(Further), ffn_norm=new(norm.RmsNorm), ffn=new(Further)))
    assert not (block.mixer_takes or block.ffn_takes or block.first_rides or block.ffn_norm_rides) and block.first_norm() is None


class Recorder:
    """A mixer or a feed-forward of a block that runs, which notes the ride it is offered."""
    in_dtype = torch.bfloat16

    def forward(self, ctx, *_):
        self.ride = ctx.ride
        ctx.stream.add_(1.0)
        return ctx.stream


class Ends(Recorder):
    adds_last = True

    def forward(self, ctx, *_):
        return super().forward(ctx)


class Twice(Ends):                               # adds to the stream behind its parent's product
    def forward(self, ctx, *_):
        super().forward(ctx)
        return ctx.stream.add_(1.0)


class TwiceAndSaysSo(Twice):
    adds_last = True


class Tanh(norm.DynamicTanh):
    def __init__(self):
        pass


class Louder(Tanh):
    def forward(self, ctx, res, out_dtype, name="normed"):
        return 2 * res.x


class Reads:                                     # (what runs here reads no rows)
    def forward(self, ctx, res, out_dtype, name="normed"):
        return res.x


class TanhThatReads(Tanh):
    """A norm that rides, for a block that runs: it says so of its own `forward`."""
    def forward(self, ctx, res, out_dtype, name="normed"):
        return res.x

    ride = norm.DynamicTanh.ride


@pytest.mark.parametrize("part, behind, rides", [(Ends, Tanh, True), (TwiceAndSaysSo, Tanh, True), (Twice, Tanh, False),
                                                 (Recorder, Tanh, False), (Ends, Louder, False), (Ends, Reads, False)])
def test_a_block_offers_the_norm_to_who_says_so(part, behind, rides):
    """A part that goes on adding to the stream, or a norm that does more than ride, is left alone: behind a mixer, and
    behind the feed-forward of the block before."""
    after = PreNormBlock(dict(mixer_norm=behind(), mixer=Recorder()))
    before = PreNormBlock(dict(mixer_norm=Reads(), mixer=Recorder(), ffn_norm=TanhThatReads(), ffn=part()))
    ctx, res = types.SimpleNamespace(stream=None, ride=None, max_seg_len=1, next_norm=after.first_norm()), Residual(torch.zeros(2, 8))
    before.forward(ctx, res, 0, True)
    assert before.mixer.ride is None             # (that mixer does not say)
    assert (before.ffn.ride is not None) == rides and (not rides or before.ffn.ride.norm is after.mixer_norm)
    alone = PreNormBlock(dict(mixer_norm=Reads(), mixer=part()))
    alone.forward(ctx, res, 0, True)
    assert (alone.mixer.ride is not None) == rides
    both = PreNormBlock(dict(mixer_norm=Reads(), mixer=part(), ffn_norm=TanhThatReads(), ffn=Recorder()))
    both.forward(ctx, res, 0, True)
    assert (both.mixer.ride is not None) == both.mixer_takes and both.ffn.ride is None
    assert res.pending is None and res.normed is None and ctx.ride is None and ctx.stream is None


def test_both_sides_of_a_pair_are_asked():
    class Side:
        adds_last = True

        def forward(self, ctx, site, owns_cache, h):
            self.ride = ctx.ride
            return ctx.stream

    class Silent(Side):
        def forward(self, ctx, site, owns_cache, h):
            self.ride = ctx.ride
            return ctx.stream

    for left, right in ((Side(), Side()), (Silent(), Side()), (Side(), Silent())):
        pair, tanh = new(mixer_pair.MixerPair), new(norm.DynamicTanh)
        pair.left, pair.right, pair.normed = left, right, False
        pair.left_takes, pair.right_takes = emits(left, "adds_last"), emits(right, "adds_last")
        ride = types.SimpleNamespace(norm=tanh, out_dtype=torch.bfloat16, rows=None)
        ctx = types.SimpleNamespace(stream=torch.zeros(2, 8), ride=ride, workspace=None)
        assert pair.forward(ctx, 0, True, torch.zeros(2, 8)) is ctx.stream
        assert (left.ride is None) == isinstance(left, Silent) and (left.ride is None or left.ride.norm is None)
        assert (right.ride is ride) == (not isinstance(right, Silent)) and (right.ride in (None, ride))


class OwnRead(norm.RmsNorm):                     # a norm from outside that reads the stream in its own way
    def _read(self, ctx, res, link, out, rows=None):
        return out.fill_(3.0)


@pytest.mark.parametrize("ffn_norm,feed,routes", [
    (norm.RmsNorm, moe.RoutedExperts, True), (norm.LayerNorm, moe.RoutedExperts, True), (OwnRead, moe.RoutedExperts, False),
    (type("OwnLinked", (norm.RmsNorm,), dict(forward_linked=lambda self, *a, **k: None)), moe.RoutedExperts, False),
    (norm.RmsNorm, type("OwnRows", (moe.RoutedExperts,), dict(_rows=lambda self, *a: None)), False),
    (norm.RmsNorm, type("OwnParts", (moe.RoutedExperts,), dict(forward_parts=None)), False), (norm.RmsNorm, ffn.SwiGlu, False)])
def test_a_router_rides_where_norm_and_mixture_say_so_of_what_they_run(ffn_norm, feed, routes):
    block = HyperBlock(dict(mixer_norm=new(norm.RmsNorm), mixer=new(attention.Attention), mixer_link=object(), ffn_norm=new(ffn_norm),
                            ffn=new(feed), ffn_link=object()))
    assert block.routes == routes


def test_a_norm_with_a_read_of_its_own_runs_behind_copies():
    ctx = types.SimpleNamespace(workspace=types.SimpleNamespace(get=lambda name, shape, dtype: torch.zeros(shape, dtype=dtype)))
    rows = new(OwnRead).forward_linked(ctx, Residual(torch.zeros(2, 4)), object(), torch.float32)
    assert torch.equal(rows, torch.full((2, 4), 3.0))

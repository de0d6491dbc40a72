"""Which norms ride with the product before them: those whose `ride` describes the `forward` they run, behind a part whose
`forward` ends with its product into the stream. Who replaces one `forward` alone gets the launches one by one."""
import types

import pytest
import torch

from imparo_amd.parts import attention, channel_delta, ffn, mixer_pair, norm, retention
from imparo_amd.parts.base import Residual
from imparo_amd.parts.block import PreNormBlock


def ride_of(part, behind):
    """The ride that a block's part is offered while it runs."""
    ctx, res, seen = types.SimpleNamespace(stream=None, ride=None), Residual(torch.zeros(2, 8)), []

    def run():
        seen.append(ctx.ride)
        return torch.zeros(2, 8)
    PreNormBlock._delta(ctx, res, run, part, (behind, torch.bfloat16))
    assert ctx.ride is None and ctx.stream is None
    return seen[0]


new = lambda cls: cls.__new__(cls)


@pytest.mark.parametrize("part", [ffn.SwiGlu, ffn.ClampedGlu, ffn.PolyNormFfn, attention.Attention, channel_delta.ChannelDelta,
                                  retention.Retention, mixer_pair.MixerPair])
def test_a_part_that_ends_with_its_product_is_offered_the_norm(part):
    tanh = new(norm.DynamicTanh)
    ride = ride_of(new(part), tanh)
    assert ride.norm is tanh and ride.rows is None
    assert ride_of(new(part), new(norm.RmsNorm)) is None


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


@pytest.mark.parametrize("mixer, behind, rides", [(Ends, Tanh, True), (TwiceAndSaysSo, Tanh, True), (Twice, Tanh, False),
                                                  (Recorder, Tanh, False), (Ends, Louder, False), (Ends, Reads, False)])
def test_a_block_offers_the_norm_to_who_says_so(mixer, behind, rides):
    """A part that goes on adding to the stream, or a norm that does more than ride, is left alone."""
    block = PreNormBlock(dict(mixer_norm=Reads(), mixer=mixer()))
    ctx, res = types.SimpleNamespace(stream=None, ride=None, max_seg_len=1, next_norm=(behind(), torch.bfloat16)), Residual(torch.zeros(2, 8))
    block.forward(ctx, res, 0, True)
    assert (block.mixer.ride is not None) == rides and res.pending is None and res.normed is None


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
        ride = types.SimpleNamespace(norm=tanh, out_dtype=torch.bfloat16, rows=None)
        ctx = types.SimpleNamespace(stream=torch.zeros(2, 8), ride=ride, workspace=None)
        assert pair.forward(ctx, 0, True, torch.zeros(2, 8)) is ctx.stream
        assert (left.ride is None) == isinstance(left, Silent) and (left.ride is None or left.ride.norm is None)
        assert (right.ride is ride) == (not isinstance(right, Silent)) and (right.ride in (None, ride))

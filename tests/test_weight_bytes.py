"""The bytes a model says its weights take: what several tensors view is counted once."""
import types

import pytest
import torch

from imparo_amd.config.plan import PartSpec
from imparo_amd.engine.model import Model
from imparo_amd.parts.channel_delta import ChannelDelta


def bytes_of(*parts):
    model = Model.__new__(Model)
    model.embedding, model.final_norm, model.head = types.SimpleNamespace(), types.SimpleNamespace(), types.SimpleNamespace()
    model.blocks = list(parts)
    return model.weight_bytes()


def test_views_count_with_what_they_view():
    whole = torch.zeros(10, 16)
    assert bytes_of(types.SimpleNamespace(w=whole)) == 640
    assert bytes_of(types.SimpleNamespace(w=whole, a=whole[:4], b=whole[4:], same=whole.view(160))) == 640
    assert bytes_of(types.SimpleNamespace(a=whole[:6], b=whole[4:]), types.SimpleNamespace(c=torch.zeros(3))) == 640 + 12
    assert bytes_of(types.SimpleNamespace(a=whole[:2], b=whole[8:], none=None, empty=torch.zeros(0))) == 256


@pytest.mark.parametrize("dtype, size", [(torch.bfloat16, 2), (torch.float32, 4)])
def test_the_channel_rules_rows_lie_in_one_matrix(dtype, size):
    H, Hk, D, E, ra, rg, taps = 2, 1, 128, 64, 16, 24, 4
    C = (2 * Hk + H) * D
    shapes = dict(q=(Hk * D, E), k=(Hk * D, E), v=(H * D, E), b=(H, E), a1=(ra, E), a2=(H * D, ra), g1=(rg, E), g2=(H * D, rg),
                  o=(E, H * D), A_log=(H,), dt_bias=(H * D,), norm=(D,))
    tensors = {f"m.{n}": torch.zeros(s, dtype=torch.bfloat16) for n, s in shapes.items()}
    tensors.update({f"m.{n}.conv": torch.zeros(shapes[n][0], taps) for n in "qkv"})
    spec = PartSpec("channel_delta", "m", dict(width=E, heads=H, kv_heads=Hk, dim=D, vdim=D, taps=taps, eps=1e-5))
    part = ChannelDelta(spec, tensors, torch.device("cpu"), dtype)
    matrices = (C + H + ra + rg) * E + 2 * H * D * (ra + rg) + E * H * D
    vectors = C * taps + H * D + H + H * D
    assert bytes_of(part) == matrices * size + vectors * 4

"""Where the inference paths that call the library by address stand back: on the CPU, where such a call would raise."""
import copy
import pickle

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad

from swin3d_amd import _lib, encoder, swin_blocks


def _operands(rows=4, k=16, n=8):
    return torch.zeros(rows, k).half(), torch.zeros(n, k).half(), torch.zeros(n).half()


def test_descriptions_do_not_stop_copies_of_the_model():
    """An average of a model's weights is a deepcopy of it, also after it was used for inference."""
    layer = nn.Linear(2, 2)
    layer._s3d_blocks = swin_blocks._Kept("key", (_lib.SwinBlock * 1)(), [])
    for other in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer))):
        assert other._s3d_blocks is None
    assert layer._s3d_blocks.key == "key"


@pytest.mark.parametrize("x,weight,bias", [
    (_operands(k=32)[0], _operands()[1], None),                  # more numbers in a row than the weight has
    (_operands()[0], _operands()[1], torch.zeros(1).half()),     # a bias that broadcasts
    (_operands()[0], _operands()[1], torch.zeros(16).half()[::2]),
    (_operands()[0], _operands()[1], torch.zeros(9).half()[1:]),  # not aligned
    (torch.zeros(4, 0).half(), torch.zeros(8, 0).half(), None),
    (_operands()[0].as_subclass(nn.Parameter), _operands()[1], None),
])
def test_linear_rows_leaves_other_operands_to_torch(x, weight, bias):
    assert swin_blocks.linear_rows(x, weight, bias) is None


def test_linear_rows_leaves_transforms_to_torch():
    x, weight, bias = _operands()
    seen = []
    torch.func.vmap(lambda row: seen.append(swin_blocks.linear_rows(row, weight, bias)) or row)(x.expand(2, 4, 16))
    with forward_ad.dual_level():
        seen.append(swin_blocks.linear_rows(x, weight, bias))
    torch.jit.trace(lambda t: seen.append(swin_blocks.linear_rows(t, weight, bias)) or t, x, check_trace=False)
    assert len(seen) >= 3 and all(s is None for s in seen)


def test_upsample_projection_keeps_its_hooks(monkeypatch):
    monkeypatch.setattr(encoder, "_fused_norm_applies", lambda feats: True)
    monkeypatch.setattr(encoder, "add_layernorm", lambda feats, pending, norm: (None, norm(feats)))
    monkeypatch.setattr(encoder, "_linear", lambda layer, x: F.linear(x, layer.weight, layer.bias))
    block, calls = nn.Sequential(nn.LayerNorm(16), nn.Linear(16, 8)), []
    block[1].register_forward_hook(lambda *_: calls.append(1))
    encoder.Upsample._norm_linear(block, torch.randn(4, 16))
    assert calls == [1]


@pytest.mark.parametrize("layer,name,value", [
    ("norm2", "eps", 1e-3), ("norm1", "normalized_shape", (4, 4)), ("attn", "fp16_mode", 0), ("attn", "scale", 0.1),
    ("attn", "num_heads", 4), ("attn", "head_dim", 4), ("attn", "dim", 8), ("attn", "cRSE", "XYZ"),
    ("attn", "table_sizes", [16] * 6), ("mlp.fc1", "out_features", 32),
])
def test_stamp_has_what_the_descriptions_follow_from(layer, name, value):
    block = encoder.SwinBlock(16, 2, 5, 4, cRSE="XYZ_RGB", fp16_mode=2)
    parts = [swin_blocks._parts(block, (encoder.SwinBlock, encoder.WindowAttention, encoder.Mlp))]
    before = swin_blocks._stamp(parts)
    assert swin_blocks._stamp(parts) == before
    setattr(block.get_submodule(layer), name, value)
    assert swin_blocks._stamp(parts) != before


def test_a_scale_set_after_a_call_reaches_the_projection():
    attn = encoder.WindowAttention(16, 5, 4, 2, cRSE="XYZ")
    with torch.no_grad():
        first = attn._prepared()[0]
        attn.scale *= 2
        second = attn._prepared()[0]
    assert torch.equal(second[:16], 2 * first[:16]) and torch.equal(second[16:], first[16:])

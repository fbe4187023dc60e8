"""The blocks of a stage in training, whose sums are left to the next norm, against the blocks one by one through torch's
layers."""
import pytest
import torch

from swin3d_amd import encoder, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hooked", [False, True])
def test_stage_gradients(hip_lib, monkeypatch, hooked):
    dev = torch.device("cuda")
    scene = synth.make_room((3.0, 3.0, 2.0), 4, 5000, seed=5)
    coords = torch.from_numpy(scene.coords).to(dev)
    signals = torch.from_numpy(synth.encoder_inputs(scene)[1].copy()).to(dev)
    torch.manual_seed(1)
    stage = encoder.Stage(48, 3, 6, 5, 4, downsample=False, cRSE="XYZ_RGB_NORM", fp16_mode=2).to(dev)
    for name, p in stage.named_parameters():
        if "table" in name or "bias" in name:
            torch.nn.init.normal_(p, std=0.1)
    feats = torch.randn(coords.shape[0], 48, device=dev, requires_grad=True)
    grad = torch.randn(coords.shape[0], 48, device=dev)
    calls = []
    if hooked:
        stage.blocks[1].register_forward_hook(lambda *_: calls.append(1))
        stage.blocks[2].norm2.register_forward_hook(lambda *_: calls.append(2))

    def run():
        with torch.autocast("cuda", dtype=torch.float16):
            out, _, _ = stage(encoder.SparseVoxels(coords, feats, 1), signals)
        return (out.feats, *torch.autograd.grad(out.feats, [feats, *stage.parameters()], grad))

    got = run()
    assert calls == ([1, 2] if hooked else [])
    monkeypatch.setattr(encoder, "trained_add_norm", lambda *_: None)
    monkeypatch.setattr(encoder, "trained_linear", lambda *_: None)
    for a, b in zip(got, run()):
        assert a.dtype == b.dtype and (a - b).norm() <= 5e-3 * b.norm()      # some ten fp16 products one after the other

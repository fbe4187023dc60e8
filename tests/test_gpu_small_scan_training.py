"""A training pass of the whole network on small scans, where fp16 activations move the gradients most: the library's
kernels against torch's operations for the same layers."""
import pytest
import torch

from swin3d_amd import encoder, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("voxels,rooms,mode", [(5000, 1, 1), (11000, 2, 2), (19000, 1, 2), (24000, 2, 1)])
def test_gradients_of_a_small_scan(hip_lib, monkeypatch, voxels, rooms, mode):
    dev = torch.device("cuda")
    scene = synth.concat_scenes([synth.make_room((3.0, 2.5, 2.0), 4, voxels // rooms, seed=voxels + b) for b in range(rooms)])
    feats, signals = (torch.from_numpy(x.copy()).to(dev) for x in synth.encoder_inputs(scene))
    coords = torch.from_numpy(scene.coords).to(dev)
    labels = torch.div(coords[:, 3], 8, rounding_mode="floor").long() % 13
    torch.manual_seed(voxels)
    model = encoder.Swin3DUNet(**encoder.SWIN3D_S, in_channels=9, cRSE="XYZ_RGB_NORM", fp16_mode=mode,
                               upsample="linear_attn", num_classes=13).to(dev).train()

    def run():
        model.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.float16):
            logits = model(encoder.SparseVoxels(coords, feats, 1), signals)
        (torch.nn.functional.cross_entropy(logits.float(), labels) * 2.0 ** 16).backward()
        return logits.detach(), [torch.cat([p.grad.reshape(-1) for p in part.parameters()]).double()
                                 for part in (model.stem_layer, *model.layers, *model.upsamples, model.classifier)]

    logits, got = run()
    monkeypatch.setattr(encoder, "trained_linear", lambda *_, **__: None)
    monkeypatch.setattr(encoder, "trained_add_norm", lambda *_: None)
    ref_logits, want = run()
    # the forward is the same to the bit; the backward's sums differ in their order, as those of two runs do (torch's
    # scatter of the interpolation adds with atomics): single roundings to fp16 on the way through some fifty layers, each
    # 2^-11 of an element at most, which leave 2 x 10^-3 of a part at the most
    assert torch.equal(logits, ref_logits)
    for g, w in zip(got, want):
        assert (g - w).norm() <= 4e-3 * w.norm() and (g - w).abs().max() <= 6e-3 * w.abs().max()

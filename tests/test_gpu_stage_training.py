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


@pytest.mark.parametrize("train", [False, True])
def test_a_block_with_an_attention_of_its_own_finds_the_unscaled_signals(hip_lib, train):
    dev = torch.device("cuda")
    scene = synth.make_room((3.0, 3.0, 2.0), 4, 3000, seed=6)
    coords = torch.from_numpy(scene.coords).to(dev)
    signals = torch.from_numpy(synth.encoder_inputs(scene)[1].copy()).to(dev)
    seen = []

    class Attention(encoder.WindowAttention):
        def forward(self, feats, attn_args):
            *_, n_coords, scaled = attn_args
            seen.append((attn_args[5], n_coords, scaled))
            return super().forward(feats, attn_args[:8])

    stage = encoder.Stage(48, 2, 6, 5, 4, downsample=False, cRSE="XYZ_RGB_NORM", fp16_mode=2).to(dev)
    feats = torch.randn(coords.shape[0], 48, device=dev)

    def run():
        with torch.set_grad_enabled(train), torch.autocast("cuda", dtype=torch.float16):
            return stage(encoder.SparseVoxels(coords, feats, 1), signals)[0].feats

    want = run()
    for block in stage.blocks:
        block.attn.__class__ = Attention
    got = run()
    assert len(seen) == 2 and (got - want).norm() <= 2e-3 * want.norm()
    local = signals[:, 1:4] - coords[:, 1:]
    for (rows, n_coords, scaled), shift in zip(seen, (0, 2)):
        inside = torch.remainder(coords[:, 1:] + shift, 5)
        assert torch.equal(n_coords, torch.cat([inside + local, signals[:, 4:]], 1)[rows.long()])
        assert torch.equal(scaled, n_coords * torch.tensor([4.0] * 3 + [8.0] * 6, device=dev))

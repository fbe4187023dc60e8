"""s3d_linear against an fp32 product at the edges of its tiles and of its dispatch, and the blocks of a stage in one call
against the blocks one by one."""
import pytest
import torch
import torch.nn.functional as F

from swin3d_amd import _lib, encoder, swin_train, synth
from swin3d_amd.swin_blocks import linear_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 16), (63, 48, 48), (65, 144, 80), (200, 72, 640),       # 64 x 64 tiles, remainders on every side
    (66000, 48, 64), (40001, 80, 48),                              # 128 x 64 and 128 x 128
    (45000, 192, 96), (33000, 144, 16),                            # 128 x 192
    (9001, 640, 80), (4100, 1152, 192),                            # several columns of tiles
])
@pytest.mark.parametrize("gelu", [False, True])
def test_linear(hip_lib, m, n, k, gelu):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w, b = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, k), (n, k), (n,)))
    w = (w.float() * k ** -0.5).half()
    ref = F.linear(x.float(), w.float(), b.float())
    for bias, want in ((b, ref), (None, ref - b.float())):
        want = F.gelu(want) if gelu else want
        got = linear_rows(x, w, bias, gelu).float()
        assert float((got - want).abs().max()) <= 1e-3 * float(want.abs().max())
        assert bool(((got - want).abs() <= 6e-4 * want.abs() + 2e-6 * float(want.abs().max()) + 6e-7).all())


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 16), (31, 40, 80), (33, 8, 256), (390, 384, 1536),      # tiles of 32 x 32 whose K eight wavefronts share, remainders on every side
    (256, 1024, 96), (257, 1024, 192), (512, 1024, 192), (513, 1024, 192),      # around 256 and 512 tiles
    (1024, 1024, 2048), (1025, 1024, 2048), (700, 640, 2560),      # long chains, up to 1024 tiles
    (100, 136, 528), (64, 96, 1040), (45, 72, 2064),               # a last chunk of 16, chunks that not every wavefront has
])
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_of_few_rows(hip_lib, m, n, k, gelu):
    test_linear(hip_lib, m, n, k, gelu)


@pytest.mark.parametrize("m,n", [(64 * tiles - 59, 64) for tiles in (575, 576, 1023, 1024)] +        # 64 x 64, 128 x 64
                         [(128 * tiles - 123, 128) for tiles in (383, 384, 447, 448, 512, 513, 639, 640, 1100)])        # ... and 128 x 128
@pytest.mark.parametrize("gelu", [False, True])
def test_linear_where_its_tiles_change(hip_lib, m, n, gelu):
    test_linear(hip_lib, m, n, 208, gelu)        # (three chunks and a quarter)


def test_gelu_of_every_number(hip_lib):
    """All finite fp16 numbers through the identity: half a place of rounding, and the approximation, which is fp32's own
    rounding and below 2^-25 where the result is too small for fp16."""
    x = torch.arange(-32768, 32768, device="cuda").to(torch.int16).view(torch.float16)
    x = torch.where(x.isfinite(), x, 0).view(-1, 16)
    got = linear_rows(x, torch.eye(16, device="cuda").half(), None, True).double()
    wide = x.double()
    want = 0.5 * wide * torch.special.erfc(-wide * 0.5 ** 0.5)
    assert bool(((got - want).abs() <= 2.0 ** -11 * 1.02 * want.abs() + 2.0 ** -25 * 1.7).all())
    assert got.isfinite().all()
    x = torch.zeros(3, 16, device="cuda").half()
    x[0, 0], x[1, 0], x[2, 0] = float("inf"), float("-inf"), float("nan")
    w = torch.ones(8, 16, device="cuda").half()
    got = linear_rows(x, w, None, True)
    assert bool((got[0] == float("inf")).all()) and bool(got[1:].isnan().all())


@pytest.mark.parametrize("m,n,k,gelu", [(300_001, 80, 16, True), (140_000, 240, 80, False), (131_137, 64, 64, True), (99_999, 192, 48, False),
                                        (70_007, 136, 144, False)])
def test_linear_of_several_tiles_a_workgroup(hip_lib, m, n, k, gelu):
    """The same rows in pieces that have a workgroup a tile: the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, device="cuda", generator=gen).half()
    w, b = torch.randn(n, k, device="cuda", generator=gen).half(), torch.randn(n, device="cuda", generator=gen).half()
    for bias in (b, None):
        whole = linear_rows(x, w, bias, gelu=gelu)
        for first in range(0, m, 4001):
            assert torch.equal(whole[first:first + 4001], linear_rows(x[first:first + 4001].clone(), w, bias, gelu=gelu))


@pytest.mark.parametrize("c", [48, 64, 80, 96, 128, 160, 192])
@pytest.mark.parametrize("m,hidden", [(1, 32), (127, 64), (129, 96), (16385, None), (40001, None)])      # one stage, two, three, the networks'; edges of 128 rows
def test_both_layers_of_an_mlp_at_once(hip_lib, c, m, hidden):
    """The bits of the layers apart."""
    hidden = hidden or 4 * c
    gen = torch.Generator(device="cuda").manual_seed(m + c)
    x, w1, b1, w2, b2 = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, c), (hidden, c), (hidden,), (c, hidden), (c,)))
    w1, w2 = (w1.float() * c ** -0.5).half(), (w2.float() * hidden ** -0.5).half()
    x[m // 2, 0], x[m // 3, 1] = float("inf"), float("nan")
    for bias1, bias2 in ((b1, b2), (None, None)):
        y = torch.empty(m + 1, c, device="cuda", dtype=torch.float16)
        y[m] = 7
        status = _lib.lib().s3d_mlp(x.data_ptr(), w1.data_ptr(), None if bias1 is None else bias1.data_ptr(), w2.data_ptr(),
                                    None if bias2 is None else bias2.data_ptr(), y.data_ptr(), m, c, hidden, _lib.stream(x.device))
        _lib.check(status, "s3d_mlp")
        # (among so many rows that no wavefronts share the sums over K)
        inner = linear_rows(torch.cat([x, x.new_zeros(40000, c)]), w1, bias1, gelu=True)[:m].contiguous()
        want = linear_rows(inner, w2, bias2, in_order=True)
        assert torch.equal(y[:m].isnan(), want.isnan()) and torch.equal(y[:m].nan_to_num(7), want.nan_to_num(7)) and bool((y[m] == 7).all())


def test_mlp_refuses_what_it_cannot_do(hip_lib):
    x = torch.zeros(64, 1024, device="cuda").half()
    for c, hidden in ((40, 32), (320, 64), (48, 48), (48, 1056)):
        assert _lib.lib().s3d_mlp(x.data_ptr(), x.data_ptr(), None, x.data_ptr(), None, x.data_ptr(), 1, c, hidden, None) < 0


def test_linear_refuses_what_it_cannot_do(hip_lib):
    x, w = torch.randn(5, 24, device="cuda").half(), torch.randn(8, 24, device="cuda").half()
    assert linear_rows(x, w, None) is None and linear_rows(x.float(), w.float(), None) is None
    assert _lib.lib().s3d_linear(x.data_ptr(), w.data_ptr(), None, x.data_ptr(), 5, 8, 24, 0, None) < 0


@pytest.mark.parametrize("heads,dim,window,mode,voxels", [(6, 8, 5, 2, 5000), (5, 16, 7, 1, 5000), (6, 8, 5, 1, 21000)])      # (both layers of the MLP at once)
def test_blocks_in_one_call_equal_single_blocks(hip_lib, heads, dim, window, mode, voxels):
    """Same launches but for the GELU (fused with fc1, which then is not rounded in between) and the products' order of
    summation; hooks and changed parameters are noticed."""
    dev = torch.device("cuda")
    scene = synth.make_room((3.0, 3.0, 2.0) if voxels < 10000 else (6.0, 5.0, 2.5), 4, voxels, seed=5)
    coords = torch.from_numpy(scene.coords).to(dev)
    assert (coords.shape[0] >= 16384) == (voxels > 10000)
    signals = torch.from_numpy(synth.encoder_inputs(scene)[1].copy()).to(dev)
    torch.manual_seed(1)
    stage = encoder.Stage(heads * dim, 3, heads, window, 4, downsample=False, cRSE="XYZ_RGB_NORM", fp16_mode=mode).to(dev).eval()
    for name, p in stage.named_parameters():
        if "table" in name or "bias" in name:
            torch.nn.init.normal_(p, std=0.1)
    feats = torch.randn(coords.shape[0], heads * dim, device=dev)
    kept, calls = feats.clone(), []

    def both():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            plan = stage.plan(coords, 1, signals)
            one, _, _ = stage(encoder.SparseVoxels(coords, feats, 1), signals, plan)
            hook = stage.blocks[1].mlp.act.register_forward_hook(lambda *_: calls.append(1))
            single, _, _ = stage(encoder.SparseVoxels(coords, feats, 1), signals, plan)
            hook.remove()
        assert (one.feats - single.feats).abs().max() <= 2e-3 * single.feats.abs().max()
        return one.feats

    first = both()
    assert len(calls) == 1 and torch.equal(feats, kept) and hasattr(stage, "_s3d_blocks")
    assert torch.equal(both(), first)
    with torch.no_grad():
        stage.blocks[2].mlp.fc2.weight.mul_(3.0)
    assert (both() - first).abs().max() > 1e-2 * first.abs().max()


def test_a_precision_set_after_a_call_is_followed(hip_lib):
    """fp16_mode 0 is not the library call's: the blocks then run one by one, the attention in fp32."""
    dev = torch.device("cuda")
    scene = synth.make_room((3.0, 3.0, 2.0), 4, 5000, seed=5)
    coords = torch.from_numpy(scene.coords).to(dev)
    signals = torch.from_numpy(synth.encoder_inputs(scene)[1].copy()).to(dev)
    torch.manual_seed(1)
    stage = encoder.Stage(48, 2, 6, 5, 4, downsample=False, cRSE="XYZ_RGB_NORM", fp16_mode=2).to(dev).eval()
    feats = torch.randn(coords.shape[0], 48, device=dev)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            return stage(encoder.SparseVoxels(coords, feats, 1), signals)[0].feats

    run()
    for block in stage.blocks:
        block.attn.fp16_mode = 0
    got = run()
    del stage._s3d_blocks
    assert torch.equal(got, run())
    assert stage._s3d_blocks.described is None


@pytest.mark.parametrize("axes,biases,shifted", [("XYZ_RGB_NORM", True, False), ("XYZ_RGB", False, True), ("XYZ", True, True)])
def test_parameters_in_one_launch_are_the_layers_copies(hip_lib, monkeypatch, axes, biases, shifted):
    """The bits of the copies that the layers make one by one; shifted: parameters at odd places of a larger buffer."""
    dev = torch.device("cuda")
    scene = synth.make_room((3.0, 3.0, 2.0), 4, 3000, seed=5)
    coords = torch.from_numpy(scene.coords).to(dev)
    signals = torch.from_numpy(synth.encoder_inputs(scene)[1].copy()).to(dev)[:, :4 + {"XYZ": 0, "XYZ_RGB": 3}.get(axes, 6)].contiguous()
    torch.manual_seed(1)
    stage = encoder.Stage(48, 2, 6, 5, 4, downsample=False, cRSE=axes, fp16_mode=2).to(dev).eval()
    for name, p in stage.named_parameters():
        torch.nn.init.normal_(p, std=0.1)
        if shifted:
            p.data = torch.cat([p.data.new_zeros(1), p.data.reshape(-1)])[1:].view(p.shape)
    if not biases:
        for block in stage.blocks:
            block.attn.qkv.bias = block.mlp.fc2.bias = None
    feats, made = torch.randn(coords.shape[0], 48, device=dev), []
    real = swin_train.packed_copies
    monkeypatch.setattr(swin_train, "packed_copies", lambda parts: made.append(real(parts)) or made[-1])

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            return stage(encoder.SparseVoxels(coords, feats, 1), signals)[0].feats

    got = run()
    assert len(made) == 2 and all(m is not None for m in made)
    run()
    assert len(made) == 2
    encoder.drop_inference_copies(stage)
    monkeypatch.setattr(swin_train, "packed_copies", lambda parts: None)
    assert torch.equal(run(), got)

"""A block in training as one node of autograd, against the nodes of its layers; the fp16 copies of its parameters."""
import ctypes

import pytest
import torch

from swin3d_amd import encoder, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,scaled,offset", [(1, 1, 0, 0), (37, 3, 11, 1), (4097, 1, 5, 0), (8, 8, 0, None), (72, 136, 24, None),
                                                     (144, 48, 48, None), (64, 64, 64, None), (1152, 384, 384, None)])
def test_half_copies(hip_lib, rows, cols, scaled, offset):
    from swin3d_amd import _lib
    dev = torch.device("cuda", 0)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    # beside an array of another kind, so that the workgroups have to be told apart
    other = torch.randn(5000, device=dev, generator=gen)
    data = torch.randn(rows * cols + 8, device=dev, generator=gen)
    data[0], data[-9:-8] = 7e4, float("nan")
    x = data[offset or 0:][:rows * cols].view(rows, cols)
    scale = 0.3535533905932738
    turned = offset is None
    half = torch.zeros(5000 + 2 * (rows * cols + 8), dtype=torch.float16, device=dev)
    same = torch.zeros(rows * cols + 8, device=dev)
    second = 5000 + -(-rows * cols // 8) * 8
    copies = (_lib.HalfCopy * 2)((5000, 1, 0, 0, -1, -1, 1.0), (rows, cols, scaled, 5000, second if turned else -1, 0, scale))
    status = _lib.lib().s3d_half_copies((ctypes.c_void_p * 2)(other.data_ptr(), x.data_ptr()), copies, 2, half.data_ptr(), same.data_ptr(),
                                        _lib.stream(dev))
    _lib.check(status, "s3d_half_copies")
    bits = lambda t: t.contiguous().view(-1).view(torch.int16)
    factor = torch.ones(rows, 1, device=dev)
    factor[:scaled] = scale
    want = (x * factor).half()
    assert torch.equal(bits(half[:5000]), bits(other.half()))
    assert torch.equal(bits(half[5000:5000 + rows * cols]), bits(want))
    assert torch.equal(same[:rows * cols].view(torch.int32), x.reshape(-1).view(torch.int32)) and not same[rows * cols:].any()
    if turned:
        assert torch.equal(bits(half[second:second + rows * cols]), bits(want.t()))


def _stage(voxels, channels, heads, window, mode, axes, seed, extent=(3.0, 3.0, 2.0), rows=None):
    dev = torch.device("cuda", 0)
    scene = synth.make_room(extent, 4, voxels, seed=seed)
    coords = torch.from_numpy(scene.coords).to(dev)[:rows]
    signals = torch.from_numpy(synth.encoder_inputs(scene)[1].copy()).to(dev)[:rows, :4 + (3 if axes == "XYZ_RGB" else 6)]
    torch.manual_seed(seed)
    stage = encoder.Stage(channels, 2, heads, window, 4, downsample=False, cRSE=axes, fp16_mode=mode).to(dev)
    for name, p in stage.named_parameters():
        if "table" in name or "bias" in name:
            torch.nn.init.normal_(p, std=0.1)
    feats = torch.randn(coords.shape[0], channels, device=dev)
    return stage, feats, (lambda f: stage(encoder.SparseVoxels(coords, f, 1), signals)[0].feats)


def _pass(stage, feats, run, wanted, seed=1, **how):
    grad = torch.randn(feats.shape, device=feats.device, generator=torch.Generator(device="cuda").manual_seed(seed))
    with torch.autocast("cuda", dtype=torch.float16):
        out = run(feats)
    return out.detach(), torch.autograd.grad(out, wanted, grad, **how)


def _nodes(t):
    seen, todo, names = set(), [t.grad_fn], []
    while todo:
        node = todo.pop()
        if node is None or node in seen:
            continue
        seen.add(node)
        names.append(node.name())
        todo += [n for n, _ in node.next_functions]
    return names


@pytest.mark.parametrize("voxels,channels,heads,window,mode,axes", [
    (5000, 48, 6, 5, 2, "XYZ_RGB_NORM"), (5001, 48, 6, 5, 1, "XYZ_RGB"), (3001, 96, 6, 7, 1, "XYZ_RGB_NORM"), (3000, 96, 6, 7, 2, "XYZ_RGB"),
    (331, 384, 24, 7, 1, "XYZ_RGB_NORM"), (7, 16, 1, 5, 2, "XYZ_RGB_NORM"), (20011, 32, 4, 5, 2, "XYZ_RGB_NORM"),
    (70001, 48, 6, 5, 2, "XYZ_RGB")])       # dense layers of several tiles a workgroup
@pytest.mark.parametrize("without", ["nothing", "biases", "some gradients"])
def test_against_the_layers_nodes(hip_lib, monkeypatch, voxels, channels, heads, window, mode, axes, without):
    stage, feats, run = _stage(voxels, channels, heads, window, mode, axes, voxels, (6.0, 5.0, 2.5) if voxels > 30000 else (3.0, 3.0, 2.0))
    assert feats.shape[0] > 0.75 * voxels
    if without == "biases":
        for block in stage.blocks:
            block.attn.qkv.bias = block.mlp.fc1.bias = None
    feats.requires_grad_(without != "some gradients")
    if without == "some gradients":
        for name, p in stage.named_parameters():
            p.requires_grad_(not any(part in name for part in ("blocks.0.attn.proj.weight", "norm2.bias", "key_xyz_table", "fc2", "blocks.1.attn.qkv")))
    wanted = [t for t in (feats, *stage.parameters()) if t.requires_grad]
    with torch.autocast("cuda", dtype=torch.float16):
        assert sum("Branches" in name for name in _nodes(run(feats))) == 2
    out, got = _pass(stage, feats, run, wanted)
    monkeypatch.setattr(encoder, "trained_branches", lambda *_: None)
    ref, want = _pass(stage, feats, run, wanted)
    assert torch.equal(out, ref)
    # the same kernels, but for GELU's derivative (fp32, some ulps, which turn single roundings to fp16 of the hidden
    # layer's gradient: 2^-11 of an element each) and the order of the tables' fp32 sums; two blocks
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and g.shape == w.shape
        assert (g - w).double().norm() <= 2 ** -11 * w.double().norm() + 1e-12


@pytest.mark.parametrize("voxels,channels,heads,mode,without", [
    (12_011, 192, 12, 1, "nothing"), (3000, 384, 24, 1, "some gradients"),      # pairs of fewer parts, in chains; pairs and single ones
    (2999, 640, 40, 1, "nothing"), (4000, 144, 9, 2, "biases")])                # too many tiles for pairs; only some have the same tiles
def test_layers_that_share_a_launch(hip_lib, monkeypatch, voxels, channels, heads, mode, without):
    test_against_the_layers_nodes(hip_lib, monkeypatch, voxels, channels, heads, 5, mode, "XYZ_RGB_NORM", without)


@pytest.mark.parametrize("rows,channels,heads,window,mode", [
    (63, 48, 6, 5, 2), (64, 48, 6, 5, 2), (811, 384, 24, 7, 1), (12_011, 192, 12, 7, 1), (65535, 48, 6, 5, 2),      # ends of the one call
    (67301, 48, 6, 5, 2)])                                                                                       # torch splits the sums of q, k, v
def test_forward_has_the_bits_of_torchs_operations(hip_lib, monkeypatch, rows, channels, heads, window, mode):
    """Products, norms, GELU and sums by torch, with the same attention between."""
    from swin3d_amd import swin_train
    stage, feats, run = _stage(rows + 8000, channels, heads, window, mode, "XYZ_RGB", 9, (8.0, 7.0, 3.0), rows)
    assert feats.shape[0] == rows
    calls = []
    monkeypatch.setattr(swin_train, "_in_one_call", lambda *a, f=swin_train._in_one_call: calls.append(f(*a)) or calls[-1])
    with torch.autocast("cuda", dtype=torch.float16):
        out = run(feats)
    assert [c is not None for c in calls] == [64 <= rows < 65536] * 2
    monkeypatch.setattr(encoder, "trained_branches", lambda *_: None)
    monkeypatch.setattr(encoder, "trained_linear", lambda *_, **__: None)
    monkeypatch.setattr(encoder, "trained_add_norm", lambda *_: None)
    monkeypatch.setattr(encoder, "add_half", lambda *_: None)
    with torch.autocast("cuda", dtype=torch.float16):
        ref = run(feats)
    names = _nodes(ref)
    assert any("AddmmBackward" in name for name in names) and not any(part in name for name in names for part in ("Branches", "_Linear", "AddNorm", "AddHalf"))
    assert torch.equal(out, ref)


def test_gradients_of_gradients_and_absent_ones(hip_lib, monkeypatch):
    stage, feats, run = _stage(900, 48, 3, 5, 2, "XYZ_RGB_NORM", seed=3)
    feats.requires_grad_()
    wanted = [feats, *stage.parameters()]
    _, plain = _pass(stage, feats, run, wanted)
    _, graph = _pass(stage, feats, run, wanted, create_graph=True)
    for g, w in zip(graph, plain):
        assert (g.detach() - w).norm() <= 2e-3 * w.norm()      # torch's products of fp16 numbers for the library's
    assert graph[0].requires_grad
    # the sum alone, without the MLP's branch: its parameters get no gradient
    block = stage.blocks[0]
    results = []
    for whole in (True, False):
        if not whole:
            monkeypatch.setattr(encoder, "trained_branches", lambda *_: None)
        seen = []
        monkeypatch.setattr(block, "forward_trained", lambda *a, f=type(block).forward_trained: seen.append(f(block, *a)) or seen[-1])
        with torch.autocast("cuda", dtype=torch.float16):
            run(feats)
        summed = seen[0][0]
        results.append(torch.autograd.grad(summed, wanted, torch.ones_like(summed), allow_unused=True))
        monkeypatch.delattr(block, "forward_trained")
    assert any(g is None for g in results[0])
    for g, w in zip(*results):
        assert (g is None) == (w is None) and (g is None or (g - w).norm() <= 2e-3 * w.norm() + 1e-12)


def test_what_steps_aside(hip_lib):
    """A layer of another kind, a hook, parameters in fp16 and a frozen block take the layers one by one."""
    def nodes(stage, run, feats):
        with torch.autocast("cuda", dtype=torch.float16):
            return sum("Branches" in name for name in _nodes(run(feats)))

    stage, feats, run = _stage(500, 48, 3, 5, 2, "XYZ_RGB", seed=4)
    assert nodes(stage, run, feats) == 2
    handle = stage.blocks[0].mlp.fc1.register_forward_hook(lambda *_: None)
    assert nodes(stage, run, feats) == 1
    handle.remove()
    stage.blocks[1].mlp.act = torch.nn.ReLU()
    assert nodes(stage, run, feats) == 1
    stage.blocks[0].attn.fp16_mode = 0
    assert nodes(stage, run, feats) == 0
    stage.blocks[0].attn.fp16_mode = 1
    assert nodes(stage, run, feats) == 1
    for p in stage.blocks[0].parameters():
        p.requires_grad_(False)
    assert nodes(stage, run, feats) == 0


@pytest.mark.parametrize("heads,mode,axes", [(3, 1, "XYZ_RGB_NORM"), (6, 2, "XYZ_RGB")])
def test_parameters_changed_between_forward_and_backward(hip_lib, monkeypatch, heads, mode, axes):
    """What the nodes of the layers let a program change in place before the backward, which then goes by the forward's values:
    every bias behind the first norm, the tables, and q, k, v's weight.  The other weights are refused."""
    stage, feats, run = _stage(1100, 48, heads, 5, mode, axes, seed=6)
    feats.requires_grad_()
    named = dict(stage.named_parameters())
    wanted = [feats, *named.values()]
    grad = torch.randn(feats.shape, device=feats.device)
    changed = [p for name, p in named.items() if "table" in name or "qkv" in name or name.endswith("bias") and "norm1" not in name]
    kept = [p.detach().clone() for p in changed]

    def gradients(change, **how):
        with torch.autocast("cuda", dtype=torch.float16):
            out = run(feats)
        if change:
            with torch.no_grad():
                for p in changed:
                    p.mul_(-1.5).add_(0.25)
        first = torch.autograd.grad(out, wanted, grad, **how)
        second = torch.autograd.grad(first[0].square().sum(), wanted, allow_unused=True) if how else ()
        with torch.no_grad():
            for p, before in zip(changed, kept):
                p.copy_(before)
        return [*first, *second]

    def close(got, want, share):
        for g, w in zip(got, want):
            assert (g is None) == (w is None) and (g is None or (g - w).norm() <= share * w.norm() + 1e-12)

    plain = gradients(False)
    close(gradients(True), plain, 1e-5)                                        # (the tables' sums are regrouped)
    whole = gradients(True, create_graph=True)
    close(whole[:len(plain)], plain, 2e-3)                                     # torch's products of fp16 numbers for the library's
    with torch.autocast("cuda", dtype=torch.float16):
        refused = run(feats)
    with torch.no_grad():
        stage.blocks[0].mlp.fc2.weight.mul_(1.0)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(refused, wanted, grad)
    # parameters that something else made go through the layers' nodes, which follow them
    module, name = stage.blocks[0].mlp.fc1, "bias"
    made = named["blocks.0.mlp.fc1.bias"] * 1.0
    monkeypatch.setitem(module._parameters, name, made)
    with torch.autocast("cuda", dtype=torch.float16):
        assert sum("Branches" in node for node in _nodes(run(feats))) == 1
    monkeypatch.undo()
    monkeypatch.setattr(encoder, "trained_branches", lambda *_: None)
    # (the second gradients: the first ones' difference and a product of the same kind again)
    close(whole, gradients(True, create_graph=True), 4e-3)


def test_gelus_derivative_at_every_fp16_number(hip_lib):
    """fc1 gives its bias, fc2 passes one row's gradient on to the whole hidden layer: fc1's bias has the derivative as its gradient."""
    hidden, values = 16384, torch.arange(-32768, 32768).to(torch.int16).view(torch.float16)
    stage, feats, run = _stage(100, 16, 1, 5, 2, "XYZ_RGB", 3)
    block, dev = stage.blocks[-1], feats.device
    block.mlp = encoder.Mlp(16, hidden).to(dev)
    torch.nn.init.zeros_(block.mlp.fc1.weight)
    torch.nn.init.zeros_(block.mlp.fc2.weight)
    block.mlp.fc2.weight.data[0] = 1
    grad = torch.zeros_like(feats)
    grad[7, 0] = 1
    for first in range(0, 65536, hidden):
        x = values[first:first + hidden]
        block.mlp.fc1.bias.data.copy_(x)
        with torch.autocast("cuda", dtype=torch.float16):
            out = run(feats)
        assert any("Branches" in name for name in _nodes(out))
        got = torch.autograd.grad(out, block.mlp.fc1.bias, grad)[0].double().cpu()
        finite, x = x.isfinite(), x.double()
        assert got[~finite].isnan().all()
        want = 0.5 * (1 + torch.erf(x / 2 ** 0.5)) + x * torch.exp(-x * x / 2) / (2 * torch.pi) ** 0.5
        # the rounding to fp16, and of fp32 before it
        assert ((got - want).abs() <= 2 ** -11 * want.abs() + 2 ** -25 + 1.5e-7)[finite].all()


def test_gelus_derivative_where_it_is_small(hip_lib):
    """From -3 down, for a gradient of 2^15, as one scaled against underflow has: relative to itself, to the last number whose product is
    a normal one in fp16, and no product of the other sign behind that."""
    hidden, dev = 4096, torch.device("cuda")
    x = torch.arange(-32768, 32768).to(torch.int16).view(torch.float16)
    x = x[(x <= -3) & (x >= -12)]
    stage, feats, run = _stage(100, 16, 1, 5, 2, "XYZ_RGB", 3)
    block = stage.blocks[-1]
    block.mlp = encoder.Mlp(16, hidden).to(dev)
    torch.nn.init.zeros_(block.mlp.fc1.weight)
    torch.nn.init.zeros_(block.mlp.fc2.weight)
    block.mlp.fc2.weight.data[0] = 1
    assert len(x) <= hidden
    block.mlp.fc1.bias.data.copy_(torch.nn.functional.pad(x.float(), (0, hidden - len(x)), value=-4.0))
    grad = torch.zeros_like(feats)
    grad[7, 0] = 2.0 ** 15
    with torch.autocast("cuda", dtype=torch.float16):
        out = run(feats)
    assert any("Branches" in name for name in _nodes(out))
    got = torch.autograd.grad(out, block.mlp.fc1.bias, grad)[0].double().cpu()[:len(x)] * 2.0 ** -15
    u = -x.double()
    phi = torch.exp(-u * u / 2) / (2 * torch.pi) ** 0.5
    want = -phi * (u - (torch.pi / 2) ** 0.5 * torch.special.erfcx(u / 2 ** 0.5))
    normal = want.abs() * 2.0 ** 15 >= 2.0 ** -14
    assert (u[normal].max() > 6) and (got <= 0).all()
    # the approximation's relative error, and the rounding to fp16
    share = torch.where(u <= 5, 1.4e-4, 1.0e-3) + 2.0 ** -11 * 1.01
    assert ((got - want).abs() <= share * want.abs())[normal].all()

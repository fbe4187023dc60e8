"""Sum, LayerNorm and their gradients in training against the same in fp64."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from swin3d_amd.fused_norm import trained_add_norm

pytestmark = pytest.mark.gpu


def _inputs(n, c, residual):
    gen = torch.Generator(device="cuda").manual_seed(n + c)
    norm = nn.LayerNorm(c).cuda()
    x = (3 * torch.randn((n, c), device="cuda", generator=gen) + 1).requires_grad_()
    res = torch.randn((n, c), device="cuda", generator=gen).half().requires_grad_() if residual else None
    with torch.no_grad():
        norm.weight.copy_(1 + 0.3 * torch.randn(c, device="cuda", generator=gen))
        norm.bias.copy_(0.3 * torch.randn(c, device="cuda", generator=gen))
    ds, dy = torch.randn((n, c), device="cuda", generator=gen), torch.randn((n, c), device="cuda", generator=gen).half()
    return norm, x, res, ds, dy


def _apply(norm, x, res):
    with torch.autocast("cuda", dtype=torch.float16):
        done = trained_add_norm(x, res, norm)
    assert done is not None and done[1].dtype == torch.float16
    return done


# every number of lanes a row and of chunks a lane, rows that fill neither, one row and more rows than a pass takes
@pytest.mark.parametrize("n,c", [(1, 4), (3, 48), (1000, 64), (9001, 80), (70001, 48), (777, 128), (4321, 160), (2049, 256),
                                 (515, 320), (300, 640), (65, 1024)])
@pytest.mark.parametrize("residual", [True, False])
@pytest.mark.parametrize("stream", [True, False])
def test_gradients(hip_lib, n, c, residual, stream):
    norm, x, res, ds, dy = _inputs(n, c, residual)
    leaves = [x, norm.weight, norm.bias] + ([res] if residual else [])
    s, y = _apply(norm, x, res)
    outs, grads = ([s, y], [ds, dy]) if stream else ([y], [dy])
    got = torch.autograd.grad(outs, leaves, grads)
    again = torch.autograd.grad(list(_apply(norm, x, res))[0 if stream else 1:], leaves, grads)
    wide = [t.detach().double().requires_grad_() for t in leaves]
    ws = wide[0] + wide[3] if residual else wide[0]
    wy = F.layer_norm(ws, (c,), wide[1], wide[2], norm.eps)
    want = torch.autograd.grad([ws, wy] if stream else [wy], wide, [g.double() for g in grads])
    assert bool(((y.double() - wy).abs() <= 2.0 ** -10 * wy.abs() + 1e-5).all())
    for g, a, w, leaf in zip(got, again, want, leaves):
        assert g.dtype == leaf.dtype and torch.equal(g, a)
        # sums in fp32 of terms whose size is that of the largest results; a rounding to fp16 for the residual
        rounding = 2.0 ** -11 if g.dtype == torch.float16 else 0.0
        assert bool(((g.double() - w).abs() <= rounding * w.abs() + 1e-5 * w.abs().max() + 1e-6).all())


def test_gradients_of_gradients(hip_lib):
    norm, x, res, ds, dy = _inputs(50, 48, True)
    s, y = _apply(norm, x, res)
    plain_s = x + res
    plain_y = F.layer_norm(plain_s, (48,), norm.weight, norm.bias, norm.eps)
    second = []
    for a, b in ((s, y), (plain_s, plain_y.half())):
        first = torch.autograd.grad([a, b], x, [ds, dy], create_graph=True)[0]
        second.append(torch.autograd.grad(first.square().sum(), [x, norm.weight]))
    for a, b in zip(*second):
        assert (a - b).abs().max() <= 1e-3 * b.abs().max()


def test_parts_that_are_not_used(hip_lib):
    norm, x, res, ds, dy = _inputs(50, 48, True)
    s, _ = _apply(norm, x, res)
    dx, dres = torch.autograd.grad(s, [x, res], ds)
    assert torch.equal(dx, ds) and torch.equal(dres, ds.half())
    _, y = _apply(norm, x.detach(), None)
    assert torch.autograd.grad(y, norm.bias, dy)[0].allclose(dy.float().sum(0), atol=1e-4)
    norm.register_forward_hook(lambda *_: None)
    with torch.autocast("cuda", dtype=torch.float16):
        assert trained_add_norm(x, res, norm) is None

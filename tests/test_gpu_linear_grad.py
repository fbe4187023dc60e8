"""s3d_linear_grad against fp32 sums at the edges of its tiles and splits, and the layer in training against F.linear."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from swin3d_amd import encoder
from swin3d_amd.linear_grad import _weight_gradients, dense_rows, trained_linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 8, 16), (63, 48, 48), (65, 144, 48), (257, 72, 640),      # one part, remainders on every side
    (1025, 240, 80), (3100, 1536, 384), (12421, 320, 320),        # several tiles and parts
    (66001, 96, 192), (199327, 48, 48),                           # as many parts as there are
    (5000, 13, 48), (700, 1, 24),                                 # columns that do not fill a load
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_weight_gradients(hip_lib, m, n, k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    dy, x = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, n), (m, k)))
    dw, db = _weight_gradients(dy, x, True, True, dtype)
    # half a unit of the result's last place for fp16, and the sums in fp32: of terms of random sign a partial sum stays
    # below 4 sqrt(m), so one of its at most m roundings (or truncations, twice that) below 2^-23 4 sqrt(m), and m of them, of
    # random sign too, below 2^-21 m sqrt(m) / sqrt(m) = 2^-21 m, where the sum of the terms' sizes is 0.64 m or more
    for got, want, terms in ((dw, dy.double().t() @ x.double(), dy.double().abs().t() @ x.double().abs()),
                             (db, dy.double().sum(0), dy.double().abs().sum(0))):
        assert bool(((got.double() - want).abs() <= (2.0 ** -11 if dtype == torch.float16 else 0.0) * want.abs() + 2.0 ** -20 * terms + 1e-7).all())
    again = _weight_gradients(dy, x, True, True, dtype)
    assert torch.equal(again[0], dw) and torch.equal(again[1], db)
    assert _weight_gradients(dy, x, False, True, dtype)[0] is None
    assert torch.equal(_weight_gradients(dy, x, True, False, dtype)[0], dw)


@pytest.mark.parametrize("m,n,k", [(1, 8, 16), (700, 48, 72), (3100, 384, 96)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gradients_inside_a_larger_buffer(hip_lib, m, n, k, dtype):
    """Wherever they lie the same bits, and nothing around them is written."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    dy, x = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, n), (m, k)))
    dw, db = _weight_gradients(dy, x, True, True, dtype)
    ws = torch.empty(hip_lib.s3d_linear_grad_workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    for offset in (0, 1, 2, 3):
        buffer = torch.full((n * k + n + 8,), -50000.0, dtype=dtype, device="cuda")
        inside = buffer[offset:offset + n * k], buffer[offset + n * k + 1:offset + n * k + 1 + n]
        assert hip_lib.s3d_linear_grad(dy.data_ptr(), x.data_ptr(), inside[0].data_ptr(), inside[1].data_ptr(), 0 if dtype == torch.float32 else 1,
                                       m, n, k, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(inside[0].view(n, k), dw) and torch.equal(inside[1], db)
        assert int((buffer == buffer[-1]).sum()) == 8


def test_weight_gradients_show_what_is_not_finite(hip_lib):
    dy, x = torch.ones(300, 48, device="cuda").half(), torch.ones(300, 64, device="cuda").half()
    dy[123, 5], x[7, 9] = float("inf"), float("nan")
    dw, db = _weight_gradients(dy, x, True, True)
    want = dy.float().t() @ x.float()
    assert torch.equal(dw.isnan(), want.isnan()) and torch.equal(dw.isinf(), want.isinf()) and db[5].isinf()


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_layer_in_training(hip_lib, bias, dtype):
    torch.manual_seed(3)
    layer = nn.Linear(96, 40, bias=bias).cuda()
    x = torch.randn(2500, 96, device="cuda").to(dtype).requires_grad_()
    leaves = [x, *layer.parameters()]
    grad = torch.randn(2500, 40, device="cuda").half()
    with torch.autocast("cuda", dtype=torch.float16):
        out, ref = encoder._linear(layer, x), F.linear(x, layer.weight, layer.bias)
        assert trained_linear(x, layer.weight, layer.bias) is not None
        layer.weight.requires_grad_(False)
        only_x = torch.autograd.grad(encoder._linear(layer, x), x, grad)[0]
        layer.weight.requires_grad_(True)
    assert type(out.grad_fn).__name__ == "_LinearBackward" and out.dtype == ref.dtype
    got, want = (torch.autograd.grad(o, leaves, grad, retain_graph=True) for o in (out, ref))
    for a, b in ((out, ref), *zip(got, want)):
        # one rounding to fp16 on either side
        assert a.dtype == b.dtype and bool(((a - b).abs() <= 2.0 ** -10 * b.abs() + 1e-4 * b.abs().max()).all())
    assert torch.equal(only_x, got[0])
    # gradients of gradients
    first = [torch.autograd.grad(o, x, grad.float().to(o.dtype).requires_grad_(), create_graph=True)[0] for o in (out, ref)]
    second = [torch.autograd.grad(f.float().square().sum(), layer.weight)[0] for f in first]
    assert (second[0] - second[1]).abs().max() <= 2e-3 * second[1].abs().max()


def test_layer_keeps_its_hooks_in_training(hip_lib):
    layer, calls = nn.Linear(32, 32).cuda(), []
    layer.register_full_backward_hook(lambda *_: calls.append(1))
    with torch.autocast("cuda", dtype=torch.float16):
        encoder._linear(layer, torch.randn(8, 32, device="cuda", requires_grad=True)).sum().backward()
    assert calls == [1]


@pytest.mark.parametrize("m", [63, 64, 811, 1563, 6250, 25013])      # torch's own, few tiles (whose K no wavefronts share), several
@pytest.mark.parametrize("n,k", [(144, 48), (48, 192), (240, 80), (384, 384), (192, 768), (384, 1536), (13, 48)])
def test_forward_of_a_layer_in_training_has_the_bits_of_torch(hip_lib, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, weight, bias = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, k), (n, k), (n,)))
    for b in (bias, None):
        assert torch.equal(dense_rows(x, weight, b), F.linear(x, weight, b))


@pytest.mark.parametrize("m,n,k,here", [
    (64, 144, 48, True), (1563, 32, 768, True), (65535, 144, 48, True), (65535, 504, 192, True), (39062, 512, 320, True), (7812, 2560, 640, True),
    (63, 144, 48, False), (67301, 144, 48, False), (131074, 48, 48, False), (199327, 192, 48, False), (264, 8, 176, False), (2000, 24, 592, False),
    (52555, 640, 160, False), (21907, 1536, 384, False), (14881, 2560, 640, False), (1563, 384, 1536, False)])
def test_forward_of_a_layer_in_training_is_here_where_torchs_bits_are(hip_lib, monkeypatch, m, n, k, here):
    """The ends of the rule, and sizes beyond it, at most of which torch splits the sums."""
    from swin3d_amd import linear_grad
    calls = []
    monkeypatch.setattr(linear_grad, "linear_rows", lambda *a, f=linear_grad.linear_rows, **how: calls.append(f(*a, **how)) or calls[-1])
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, weight, bias = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, k), (n, k), (n,)))
    assert torch.equal(dense_rows(x, weight, bias), F.linear(x, weight, bias))
    assert [c is not None for c in calls] == [True] * here


def _rows_and_gelu(x, weight, bias):
    from swin3d_amd import _lib
    y, gelu = (torch.full((x.shape[0], weight.shape[0]), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    status = _lib.lib().s3d_linear_in_order(x.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), gelu.data_ptr(),
                                            x.shape[0], weight.shape[0], x.shape[1], _lib.stream(x.device))
    _lib.check(status, "s3d_linear_in_order")
    return y, gelu


def _same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7), b.nan_to_num(7))      # (torch has zeros of either sign)


def test_gelu_of_a_training_forward_has_the_bits_of_torch(hip_lib):
    """Of every fp16 number, infinities and NaN among them."""
    values = torch.arange(-32768, 32768, device="cuda").to(torch.int16).view(torch.float16)
    x, weight = (torch.zeros(s, dtype=torch.float16, device="cuda") for s in ((65536, 16), (8, 16)))
    x[:, 0], weight[:, 0] = values, 1
    y, gelu = _rows_and_gelu(x, weight, None)
    assert torch.equal(y[:, 3].isnan(), values.isnan()) and torch.equal(y[:, 3].nan_to_num(7), values.nan_to_num(7))
    assert _same(gelu, F.gelu(y))


@pytest.mark.parametrize("m,n,k", [(1, 8, 16), (63, 64, 48), (129, 72, 64), (16387, 192, 48), (16385, 384, 96), (70001, 72, 16)])      # each tile, and its edges
def test_gelu_beside_a_layers_rows(hip_lib, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m)
    x, weight, bias = (torch.randn(s, device="cuda", generator=gen).half() for s in ((m, k), (n, k), (n,)))
    y, gelu = _rows_and_gelu(x, weight, bias)
    from swin3d_amd.swin_blocks import linear_rows
    assert torch.equal(y, linear_rows(x, weight, bias, in_order=True)) and _same(gelu, F.gelu(y))

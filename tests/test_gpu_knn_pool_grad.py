"""The gradient of the maximum over neighbours against autograd of the tensor statement."""
import pytest
import torch

from swin3d_amd.sparse_dl.knn import KNNMaxPool, knn_max_pool

pytestmark = pytest.mark.gpu


def _inputs(nq, k, ns, c, dtype):
    gen = torch.Generator(device="cuda").manual_seed(nq + k + ns + c)
    idx = torch.randint(-1, ns, (nq, k), device="cuda", generator=gen, dtype=torch.int32)      # -1: reads row 0
    feats = torch.randint(-8, 8, (ns, c), device="cuda", generator=gen).to(dtype) / 4          # many shared maxima
    return idx, feats, torch.randn((nq, c), device="cuda", generator=gen).to(dtype)


def _statement(idx, feats):
    return feats[idx.reshape(-1).long().clamp(min=0)].view(*idx.shape, feats.shape[1]).amax(1)


@pytest.mark.parametrize("nq,k,ns,c", [(1, 1, 1, 8), (3, 16, 2, 48), (500, 16, 2000, 96), (777, 3, 4000, 13), (4000, 16, 300, 40),
                                       (257, 64, 999, 24), (2000, 9, 1, 16)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gradient(hip_lib, nq, k, ns, c, dtype):
    idx, feats, grad = _inputs(nq, k, ns, c, dtype)
    feats.requires_grad_()
    out = KNNMaxPool.apply(idx, feats)
    got, again = (torch.autograd.grad(KNNMaxPool.apply(idx, feats), feats, grad)[0] for _ in range(2))
    assert torch.equal(out, _statement(idx, feats)) and torch.equal(got, again) and got.dtype == dtype
    # the shares as they are rounded, added up in fp64
    rows = idx.reshape(-1).long().clamp(min=0)
    held = feats.detach()[rows].view(nq, k, c) == out.detach().unsqueeze(1)
    share = (grad.float() / held.sum(1)).to(dtype).double()
    want = torch.zeros((ns, c), dtype=torch.float64, device="cuda").index_add_(0, rows, (share.unsqueeze(1) * held).reshape(-1, c))
    last = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -23
    assert bool(((got.double() - want).abs() <= last * want.abs() + 1e-30).all())


def test_gradient_of_the_gradient(hip_lib):
    idx, feats, grad = _inputs(40, 16, 100, 8, torch.float32)
    feats.requires_grad_(), grad.requires_grad_()
    second = []
    for out in (KNNMaxPool.apply(idx, feats), _statement(idx, feats)):
        first = torch.autograd.grad(out, feats, grad, create_graph=True)[0]
        second.append(torch.autograd.grad(first.square().sum(), grad)[0])
    assert torch.allclose(second[0], second[1], atol=1e-5)


def test_what_is_not_a_number_shows(hip_lib):
    idx, feats, grad = _inputs(50, 16, 100, 8, torch.float16)
    feats[7, 3] = float("nan")
    assert torch.equal(knn_max_pool(idx, feats).isnan(), _statement(idx, feats).isnan())
    feats.requires_grad_()
    got, want = (torch.autograd.grad(out, feats, grad)[0] for out in (KNNMaxPool.apply(idx, feats), _statement(idx, feats)))
    assert want.isnan().any() and torch.equal(got.isnan(), want.isnan())

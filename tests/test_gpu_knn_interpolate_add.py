"""The upsample's sum of skip features and interpolated ones (fp16 in, fp32 out) in one kernel, and its gradients, against the
two steps it replaces."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _neighbours(nq, ns, k, seed):
    """A list with an empty place or two where there is a second batch element of fewer sources than k."""
    import swin3d_amd
    rng = np.random.default_rng(seed)
    t = lambda *shape: torch.from_numpy((rng.random(shape) * 6).astype(np.float32)).cuda()
    few = min(2, ns - 1)
    ends = lambda n, last: torch.tensor([n - last, n], dtype=torch.int32).cuda()
    idx, dist2 = swin3d_amd.knn_query(k, t(ns, 3), t(nq, 3), ends(ns, few), ends(nq, min(5, nq - 1)))
    return idx, dist2


@pytest.mark.parametrize("nq,ns,channels,k", [(1, 3, 4, 3), (700, 300, 48, 3), (700, 300, 36, 3), (1023, 257, 192, 3), (65, 40, 8, 1), (300, 90, 20, 7)])
def test_sum_and_gradients(hip_lib, nq, ns, channels, k):
    import swin3d_amd
    from swin3d_amd.sparse_dl.knn import KNNInterpolateAdd, interpolate_add_applies
    idx, dist2 = _neighbours(nq, ns, k, channels)
    gen = torch.Generator("cuda").manual_seed(nq)
    feat, skip = (torch.randn((n, channels), device="cuda", generator=gen).half().requires_grad_() for n in (ns, nq))
    dout = torch.randn((nq, channels), device="cuda", generator=gen)
    assert interpolate_add_applies(idx, dist2, feat, skip) and not interpolate_add_applies(idx, dist2, feat[:, :3], skip[:, :3])
    out = KNNInterpolateAdd.apply(idx, dist2, feat, skip)
    assert torch.equal(out, skip + swin3d_amd.KNNInterpolate.apply(idx, dist2, feat.float()))
    got = torch.autograd.grad(out, (feat, skip), dout)
    assert torch.equal(got[1], dout.half())
    weight = torch.where(idx >= 0, 1 / (dist2.double().sqrt() + 1e-8), 0.0)
    weight = weight / weight.sum(1, keepdim=True)
    ref, size = (torch.zeros((ns, channels), dtype=torch.float64, device="cuda") for _ in range(2))
    for i in range(k):
        rows, share = idx[:, i].clamp(min=0).long(), weight[:, i:i + 1]
        ref.index_add_(0, rows, dout.double() * share)
        size.index_add_(0, rows, (dout.double() * share).abs())
    # a share of dout is rounded some ten times, and a sum of n of them up to n times: 2^-24 each of the terms' sizes; the result
    # to fp16
    most = int(torch.bincount(idx[idx >= 0].long()).max())
    assert bool(((got[0].double() - ref).abs() <= 2.0 ** -11 * ref.abs() + (10 + most) * 2.0 ** -24 * size + 2.0 ** -25).all())
    # with a graph of the gradients: by operations that have one
    (again,) = torch.autograd.grad(KNNInterpolateAdd.apply(idx, dist2, feat, skip), feat, dout.requires_grad_(), create_graph=True)
    assert again.requires_grad and bool(((again.double() - ref).abs() <= 2.0 ** -11 * ref.abs() + (10 + most) * 2.0 ** -24 * size + 2.0 ** -25).all())


@pytest.mark.parametrize("channels", [124, 128, 132, 136, 252, 256, 260])      # a whole row in lanes side by side, half a row, a quarter
def test_gradients_where_the_rows_are_halved(hip_lib, channels):
    test_sum_and_gradients(hip_lib, 515, 130, channels, 3)


@pytest.mark.parametrize("add", [False, True])
def test_gradients_in_a_fixed_order_where_a_program_asks_for_it(hip_lib, add):
    """Under torch.use_deterministic_algorithms the gradient is that of index_add, the same bits on every call: here with some
    500 terms a sum of sizes apart, whose order shows."""
    import swin3d_amd
    from swin3d_amd.sparse_dl.knn import KNNInterpolateAdd
    nq, ns, channels, k = 20_000, 128, 64, 3
    idx, dist2 = _neighbours(nq, ns, k, 5)
    gen = torch.Generator("cuda").manual_seed(6)
    feat, skip = (torch.randn((n, channels), device="cuda", generator=gen).half().requires_grad_() for n in (ns, nq))
    wide = feat.detach().float().requires_grad_()
    dout = torch.randn((nq, channels), device="cuda", generator=gen) * 2.0 ** torch.randint(-12, 12, (nq, 1), device="cuda", generator=gen)

    def grads():
        if add:
            return torch.autograd.grad(KNNInterpolateAdd.apply(idx, dist2, feat, skip), (feat, skip), dout)
        return torch.autograd.grad(swin3d_amd.KNNInterpolate.apply(idx, dist2, wide), (wide,), dout)

    rows = idx.clamp(min=0).long()
    weight = torch.where(idx >= 0, 1.0 / (torch.sqrt(dist2) + 1e-8), torch.zeros_like(dist2))
    weight = weight / weight.sum(dim=1, keepdim=True).clamp_min(1e-30)
    torch.use_deterministic_algorithms(True)
    try:
        want = torch.zeros((ns, channels), device="cuda")
        for i in range(k):
            want.index_add_(0, rows[:, i], dout * weight[:, i:i + 1])
        for _ in range(8):
            got = grads()
            assert torch.equal(got[0], want.half() if add else want)
    finally:
        torch.use_deterministic_algorithms(False)


def test_gradients_of_neighbours_beyond_any_distance(hip_lib):
    """Infinite distances have no share, also where a query has no other neighbours; NaN makes NaN."""
    import swin3d_amd
    idx = torch.tensor([[0, 1, 2], [1, 2, 3], [2, 3, 4], [4, 5, -1], [-1, -1, -1], [6, 7, 5]], dtype=torch.int32, device="cuda")
    dist2 = torch.rand((6, 3), device="cuda") + 0.5
    dist2[1, 0], dist2[2], dist2[3, :2], dist2[5, 1] = float("inf"), float("inf"), float("inf"), float("nan")
    feat = torch.randn((8, 8), device="cuda").requires_grad_()
    dout = torch.randn((6, 8), device="cuda")
    (got,) = torch.autograd.grad(swin3d_amd.KNNInterpolate.apply(idx, dist2, feat), feat, dout)
    (want,) = torch.autograd.grad(swin3d_amd.KNNInterpolate.apply(idx, dist2, feat), feat, dout.requires_grad_(), create_graph=True)
    assert torch.equal(got.isnan(), want.isnan()) and int(got.isnan().any(1).sum()) == 3      # the sources of the last query
    assert bool(((got - want).abs() <= 2.0 ** -20 * (1 + want.abs()))[~want.isnan()].all())
    assert not got[4].any()

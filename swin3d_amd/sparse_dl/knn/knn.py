"""K-nearest-neighbour operator on the swin3d_amd HIP library.

Same Python surface as Swin3D/sparse_dl/knn/knn.py:9-26: KNN.apply(K, src_xyz, query_xyz,
src_offset, query_offset) -> (idx int32 [Nq,K], euclidean dist fp32 [Nq,K]); offsets are
cumulative END positions of the batch segments.  Result order: ascending (distance, source
row); segments with fewer than K sources are padded with row -1.
"""
import torch
from torch.autograd.function import Function

from ... import _lib
from ...swin_blocks import data_only


def knn_query(K, src_xyz, query_xyz, src_offset, query_offset, cell_size=0.0, squared=True, strided=False):
    """-> (idx int32 [Nq,K], SQUARED distances fp32 [Nq,K], or the distances with squared=False).  cell_size <= 0: chosen
    from the data.  strided: the coordinates may be columns of a wider matrix (with squared distances)."""
    K = int(K)
    if not 1 <= K <= _lib.KNN_KMAX:
        raise ValueError(f"K must be in 1..{_lib.KNN_KMAX}, got {K}")
    for name, t in (("src_xyz", src_xyz), ("query_xyz", query_xyz)):
        if not t.is_cuda:
            raise RuntimeError(f"{name} must be a CUDA (HIP) tensor")
        if not (t.is_contiguous() or (strided and squared and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) >= 3)):
            raise RuntimeError(f"{name} must be contiguous")
        if t.dtype != torch.float32 or t.dim() != 2 or t.shape[1] != 3:
            raise ValueError(f"{name} must be float32 [n,3], got {t.dtype} {tuple(t.shape)}")
    dev = query_xyz.device
    if src_xyz.device != dev:
        raise RuntimeError("src_xyz and query_xyz must be on the same device")
    offs = []
    for name, t in (("src_offset", src_offset), ("query_offset", query_offset)):
        if not isinstance(t, torch.Tensor):
            t = torch.as_tensor(t)
        if t.dtype not in (torch.int32, torch.int64) or t.dim() != 1:
            raise TypeError(f"{name} must be a 1-D int32/int64 tensor")
        offs.append(t.to(device=dev, dtype=torch.int32).contiguous())
    src_offset, query_offset = offs
    if src_offset.numel() != query_offset.numel() or src_offset.numel() == 0:
        raise ValueError("src_offset and query_offset must have the same non-zero length")
    ns, nq, b = src_xyz.shape[0], query_xyz.shape[0], src_offset.numel()
    idx = torch.empty((nq, K), dtype=torch.int32, device=dev)
    dist2 = torch.empty((nq, K), dtype=torch.float32, device=dev)
    lib = _lib.lib()
    with _lib.on(dev):
        ws_bytes = lib.s3d_knn_workspace_bytes(ns, nq, b)
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        stream = _lib.stream(dev)
        fn = lib.s3d_knn if squared else lib.s3d_knn_distances
        if not (src_xyz.is_contiguous() and query_xyz.is_contiguous()):
            status = lib.s3d_knn_strided(K, src_xyz.data_ptr(), src_xyz.stride(0) if ns > 1 else 3, ns, query_xyz.data_ptr(),
                                         query_xyz.stride(0) if nq > 1 else 3, nq, src_offset.data_ptr(), query_offset.data_ptr(), b,
                                         idx.data_ptr(), dist2.data_ptr(), float(cell_size), workspace.data_ptr(), ws_bytes, stream)
        else:
            status = fn(K, src_xyz.data_ptr(), ns, query_xyz.data_ptr(), nq,
                    src_offset.data_ptr(), query_offset.data_ptr(), b, idx.data_ptr(),
                    dist2.data_ptr(), float(cell_size), workspace.data_ptr(), ws_bytes,
                    stream)
    _lib.check(status, "s3d_knn")
    return idx, dist2


class KNN(Function):
    # edge of the bucketing grid in xyz units; 0 lets the library choose from the data
    cell_size = 0.0

    @staticmethod
    def forward(ctx, K, src_xyz, query_xyz, src_offset, query_offset):
        idx, dist = knn_query(K, src_xyz, query_xyz, src_offset, query_offset, KNN.cell_size, squared=False)
        ctx.mark_non_differentiable(idx, dist)
        return idx, dist


_FEAT_DTYPE = {torch.float32: 0, torch.float16: 1}


def knn_interpolate(idx, dist2, src_feat):
    """Inverse-distance interpolation of src_feat [Ns,C] at the queries of a knn_query result
    (idx int32 [Nq,K], SQUARED distances fp32 [Nq,K]) -> [Nq,C] in the dtype of src_feat
    (Swin3D/modules/swin3d_layers.py:65-72 in one kernel; padded slots carry no weight)."""
    if not (idx.is_cuda and dist2.is_cuda and src_feat.is_cuda):
        raise RuntimeError("idx, dist2 and src_feat must be CUDA (HIP) tensors")
    if idx.dtype != torch.int32 or dist2.dtype != torch.float32 or idx.shape != dist2.shape or idx.dim() != 2:
        raise ValueError("idx must be int32 [Nq,K] and dist2 float32 [Nq,K]")
    if src_feat.dim() != 2 or src_feat.dtype not in _FEAT_DTYPE:
        raise ValueError(f"src_feat must be float16/float32 [Ns,C], got {src_feat.dtype} {tuple(src_feat.shape)}")
    idx, dist2, src_feat = idx.contiguous(), dist2.contiguous(), src_feat.contiguous()
    nq, k = idx.shape
    ns, c = src_feat.shape
    out = torch.empty((nq, c), dtype=src_feat.dtype, device=src_feat.device)
    with _lib.on(src_feat.device):
        stream = _lib.stream(src_feat.device)
        status = _lib.lib().s3d_knn_interpolate(idx.data_ptr(), dist2.data_ptr(), k, nq, src_feat.data_ptr(), ns, c,
                                                _FEAT_DTYPE[src_feat.dtype], out.data_ptr(), stream)
    _lib.check(status, "s3d_knn_interpolate")
    return out


def knn_max_pool(idx, src_feat):
    """Channel-wise maximum of src_feat [Ns,C] over the K nearest sources of every query (idx int32 [Nq,K] of a
    knn_query result) -> [Nq,C] in the dtype of src_feat: the gather + max of the KNN downsample
    (Swin3D/modules/swin3d_layers.py:292-312) without the [Nq,K,C] intermediate.  Padded slots (row -1) read
    row 0, as the clamped gather does.  No autograd: KNNMaxPool has it."""
    return _max_pool(idx, src_feat, src_feat.dtype)


def _max_pool(idx, src_feat, dtype):
    """knn_max_pool in `dtype`: that of src_feat, or float32."""
    if not (idx.is_cuda and src_feat.is_cuda):
        raise RuntimeError("idx and src_feat must be CUDA (HIP) tensors")
    if idx.dtype != torch.int32 or idx.dim() != 2:
        raise ValueError("idx must be int32 [Nq,K]")
    if src_feat.dim() != 2 or src_feat.dtype not in _FEAT_DTYPE:
        raise ValueError(f"src_feat must be float16/float32 [Ns,C], got {src_feat.dtype} {tuple(src_feat.shape)}")
    idx, src_feat = idx.contiguous(), src_feat.contiguous()
    nq, k = idx.shape
    ns, c = src_feat.shape
    out = torch.empty((nq, c), dtype=dtype, device=src_feat.device)
    with _lib.on(src_feat.device):
        stream = _lib.stream(src_feat.device)
        if dtype == src_feat.dtype:
            status = _lib.lib().s3d_knn_max_pool(idx.data_ptr(), k, nq, src_feat.data_ptr(), ns, c,
                                                 _FEAT_DTYPE[src_feat.dtype], out.data_ptr(), stream)
        else:
            status = _lib.lib().s3d_knn_max_pool_widened(idx.data_ptr(), k, nq, src_feat.data_ptr(), ns, c, out.data_ptr(), stream)
    _lib.check(status, "s3d_knn_max_pool")
    return out


class KNNMaxPool(Function):
    """Differentiable (w.r.t. the features) knn_max_pool: KNNMaxPool.apply(idx, src_feat).  Rows that share a maximum share
    its gradient, as under torch's amax."""

    @staticmethod
    def forward(ctx, idx, src_feat):
        idx, src_feat = idx.contiguous(), src_feat.contiguous()
        out = knn_max_pool(idx, src_feat)
        ctx.save_for_backward(idx, src_feat, out)
        return out

    @staticmethod
    def backward(ctx, dout):
        idx, src_feat, out = ctx.saved_tensors
        if torch.is_grad_enabled() or not data_only(dout) or dout.dtype != src_feat.dtype:
            # a graph of the gradient is wanted, or something follows it: operations that have one
            rows = idx.reshape(-1).long().clamp(min=0)
            gathered = src_feat[rows].view(*idx.shape, src_feat.shape[1])
            held = (gathered == out.unsqueeze(1)).to(dout.dtype)
            given = (dout / held.sum(1)).unsqueeze(1) * held
            return None, torch.zeros_like(src_feat).index_add(0, rows, given.reshape(-1, src_feat.shape[1]).to(src_feat.dtype))
        dout = dout.contiguous()
        (nq, k), (ns, c) = idx.shape, src_feat.shape
        grad = torch.empty_like(src_feat)
        code = _FEAT_DTYPE[src_feat.dtype]
        lib = _lib.lib()
        with _lib.on(src_feat.device):
            ws_bytes = lib.s3d_knn_max_pool_grad_workspace_bytes(nq, k, ns, c, code)
            workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=src_feat.device)
            status = lib.s3d_knn_max_pool_grad(idx.data_ptr(), k, nq, src_feat.data_ptr(), ns, c, code, out.data_ptr(),
                                               dout.data_ptr(), grad.data_ptr(), workspace.data_ptr(), ws_bytes,
                                               _lib.stream(src_feat.device))
        _lib.check(status, "s3d_knn_max_pool_grad")
        return None, grad


def _interpolate_grads(idx, dist2, grad_out, num_src, need_src, need_skip):
    """Gradients of the interpolation (fp32) and of fp16 features beside it for grad_out in fp32, by one launch behind a fill."""
    grad_out = grad_out.contiguous()
    nq, c = grad_out.shape
    grad_src = torch.zeros((num_src, c), dtype=torch.float32, device=grad_out.device) if need_src else None
    grad_skip = torch.empty((nq, c), dtype=torch.float16, device=grad_out.device) if need_skip else None
    with _lib.on(grad_out.device):
        status = _lib.lib().s3d_knn_interpolate_grad(idx.data_ptr(), dist2.data_ptr(), idx.shape[1], nq, grad_out.data_ptr(), num_src, c,
                                                     None if grad_src is None else grad_src.data_ptr(),
                                                     None if grad_skip is None else grad_skip.data_ptr(), _lib.stream(grad_out.device))
    _lib.check(status, "s3d_knn_interpolate_grad")
    return grad_src, grad_skip


def _native_grads(idx, dist2, grad_out, num_src):
    """The library's kernel has these gradients: no graph of them is wanted, nothing follows them, it takes the types, and any
    order of the additions will do (torch's index_add has a fixed one for programs that ask for it)."""
    return (not torch.is_grad_enabled() and not torch.are_deterministic_algorithms_enabled() and data_only(grad_out) and grad_out.is_cuda and grad_out.dtype == torch.float32
            and grad_out.shape[1] % 4 == 0 and grad_out.shape[1] > 0 and num_src > 0
            and idx.is_contiguous() and dist2.is_contiguous() and idx.dtype == torch.int32)


class KNNInterpolate(Function):
    """Differentiable (w.r.t. the features) inverse-distance interpolation; the forward is the fused
    HIP kernel, the backward adds the weighted output gradient to the sources' rows."""

    @staticmethod
    def forward(ctx, idx, dist2, src_feat):
        ctx.save_for_backward(idx, dist2)
        ctx.num_src = src_feat.shape[0]
        return knn_interpolate(idx, dist2, src_feat)

    @staticmethod
    def backward(ctx, grad_out):
        idx, dist2 = ctx.saved_tensors
        if _native_grads(idx, dist2, grad_out, ctx.num_src):
            return None, None, _interpolate_grads(idx, dist2, grad_out, ctx.num_src, True, False)[0]
        valid = idx >= 0
        weight = torch.where(valid, 1.0 / (torch.sqrt(dist2) + 1e-8), torch.zeros_like(dist2))
        weight = weight / weight.sum(dim=1, keepdim=True).clamp_min(1e-30)
        grad_src = torch.zeros((ctx.num_src, grad_out.shape[1]), dtype=torch.float32, device=grad_out.device)
        rows = idx.clamp(min=0).long()
        for i in range(idx.shape[1]):
            grad_src.index_add_(0, rows[:, i], grad_out.float() * weight[:, i:i + 1])
        return None, None, grad_src.to(grad_out.dtype)


class KNNInterpolateAdd(Function):
    """skip + KNNInterpolate of the features, both fp16, in fp32: an upsample's sum in one kernel.  The caller has checked
    interpolate_add_applies."""

    @staticmethod
    def forward(ctx, idx, dist2, src_feat, skip):
        ctx.save_for_backward(idx, dist2)
        ctx.num_src = src_feat.shape[0]
        (nq, k), c = idx.shape, src_feat.shape[1]
        out = torch.empty((nq, c), dtype=torch.float32, device=src_feat.device)
        with _lib.on(src_feat.device):
            status = _lib.lib().s3d_knn_interpolate_add(idx.data_ptr(), dist2.data_ptr(), k, nq, src_feat.data_ptr(), src_feat.shape[0], c,
                                                        skip.data_ptr(), out.data_ptr(), _lib.stream(src_feat.device))
        _lib.check(status, "s3d_knn_interpolate_add")
        return out

    @staticmethod
    def backward(ctx, grad_out):
        idx, dist2 = ctx.saved_tensors
        _, _, need_src, need_skip = ctx.needs_input_grad
        if _native_grads(idx, dist2, grad_out, ctx.num_src):
            grad_src, grad_skip = _interpolate_grads(idx, dist2, grad_out, ctx.num_src, need_src, need_skip)
            return None, None, None if grad_src is None else grad_src.half(), grad_skip
        grad_src = KNNInterpolate.backward(ctx, grad_out)[2].half() if need_src else None
        return None, None, grad_src, grad_out.half() if need_skip else None


def interpolate_add_applies(idx, dist2, src_feat, skip):
    """KNNInterpolateAdd can stand in for skip + KNNInterpolate of src_feat.float()."""
    return (all(data_only(t) and t.is_cuda and t.device == idx.device and t.is_contiguous() for t in (idx, dist2, src_feat, skip))
            and src_feat.dtype == skip.dtype == torch.float16 and idx.dtype == torch.int32 and dist2.dtype == torch.float32
            and src_feat.dim() == skip.dim() == 2 and idx.dim() == 2 and skip.shape == (idx.shape[0], src_feat.shape[1])
            and src_feat.shape[0] > 0 and src_feat.shape[1] > 0 and src_feat.shape[1] % 4 == 0
            and src_feat.data_ptr() % 16 == 0 and skip.data_ptr() % 16 == 0)

"""Residual add fused with LayerNorm (HIP kernel s3d_add_layernorm) for the Swin block around the
attention operator (Swin3D/modules/swin3d_layers.py:617-623)."""
import torch
import torch.nn as nn
from torch.autograd.function import Function

from . import _lib
from .swin_blocks import data_only, followed, plain

_DTYPE_CODE = {torch.float32: _lib.S3D_DTYPE_F32, torch.float16: _lib.S3D_DTYPE_F16}


def add_layernorm(x, residual, norm, out_dtype=torch.float16, inplace=False):
    """(x + residual, LayerNorm(x + residual)) for x fp32 [N,C] on the GPU and `norm` a torch.nn.LayerNorm over C.

    residual   fp16 / fp32 [N,C] or None (then the first result is x itself)
    out_dtype  dtype of the normalised rows (fp16: what the next GEMM reads under autocast)
    inplace    write the sum back into x instead of a new tensor
    No autograd: for inference, or inside torch.no_grad().
    """
    if not x.is_cuda or x.dtype != torch.float32 or x.dim() != 2:
        raise ValueError(f"x must be a float32 [N,C] CUDA (HIP) tensor, got {x.dtype} {tuple(x.shape)} on {x.device}")
    n, c = x.shape
    if tuple(norm.normalized_shape) != (c,) or norm.weight is None or norm.bias is None:
        raise ValueError("norm must be an affine LayerNorm over the channel axis")
    if out_dtype not in _DTYPE_CODE:
        raise ValueError(f"out_dtype {out_dtype} (float16 or float32)")
    x = x.contiguous()
    res_ptr, res_code = None, 0
    summed = x
    if residual is not None:
        if residual.shape != x.shape or residual.dtype not in _DTYPE_CODE or residual.device != x.device:
            raise ValueError("residual must be float16/float32 of x's shape on x's device")
        residual = residual.contiguous()
        res_ptr, res_code = residual.data_ptr(), _DTYPE_CODE[residual.dtype]
        summed = x if inplace else torch.empty_like(x)
    y = torch.empty((n, c), dtype=out_dtype, device=x.device)
    gamma, beta = norm.weight.detach().float().contiguous(), norm.bias.detach().float().contiguous()
    with _lib.on(x.device):
        stream = _lib.stream(x.device)
        status = _lib.lib().s3d_add_layernorm(x.data_ptr(), res_ptr, res_code, gamma.data_ptr(), beta.data_ptr(),
                                             float(norm.eps), summed.data_ptr() if residual is not None else None,
                                             y.data_ptr(), _DTYPE_CODE[out_dtype], n, c, stream)
    _lib.check(status, "s3d_add_layernorm")
    return summed, y


def train_add_layernorm(x, residual, weight, bias, eps):
    """(x + residual, LayerNorm of it in fp16) for dense 16-byte aligned fp32 rows and a branch in fp16 or None, with the bits of
    torch's operations: a rounding of the mean elsewhere in fp32 moves single fp16 roundings of the rows, and with them the
    gradients of an encoder on scans of 20,000 voxels by a fiftieth (see linear_grad.py)."""
    summed = x if residual is None else torch.empty_like(x)
    y = torch.empty_like(x, dtype=torch.float16)
    with _lib.on(x.device):
        status = _lib.lib().s3d_train_add_layernorm(x.data_ptr(), None if residual is None else residual.data_ptr(), weight.data_ptr(),
                                                    bias.data_ptr(), eps, None if residual is None else summed.data_ptr(), y.data_ptr(),
                                                    x.shape[0], x.shape[1], _lib.stream(x.device))
    _lib.check(status, "s3d_train_add_layernorm")
    return summed, y


def add_half(x, residual):
    """x + residual for fp32 rows and a branch in fp16, with their gradients where they are followed; None where the kernel does
    not take them."""
    if followed() or not (x.is_cuda and type(x) is type(residual) is torch.Tensor and x.dtype == torch.float32 and residual.dtype == torch.float16
                          and x.device == residual.device and x.shape == residual.shape and x.is_contiguous() and residual.is_contiguous()
                          and x.numel() % 4 == 0 and (x.data_ptr() | residual.data_ptr()) % 16 == 0):
        return None
    return _AddHalf.apply(x, residual) if torch.is_grad_enabled() and (x.requires_grad or residual.requires_grad) else _added_half(x, residual)


def _added_half(x, residual):
    out = torch.empty_like(x)
    with _lib.on(x.device):
        status = _lib.lib().s3d_add_half(x.data_ptr(), residual.data_ptr(), out.data_ptr(), x.numel(), _lib.stream(x.device))
    _lib.check(status, "s3d_add_half")
    return out


class _AddHalf(Function):
    @staticmethod
    def forward(ctx, x, residual):
        return _added_half(x, residual)

    @staticmethod
    def backward(ctx, grad):
        return grad, grad.to(torch.float16) if ctx.needs_input_grad[1] else None


class _AddNorm(Function):
    """(x + residual, LayerNorm of it in fp16); x itself in the first place without a residual."""

    @staticmethod
    def forward(ctx, x, residual, weight, bias, norm):
        ctx.set_materialize_grads(False)
        summed, y = train_add_layernorm(x, residual, weight, bias, norm.eps)
        ctx.save_for_backward(summed, weight)
        ctx.eps, ctx.residual = norm.eps, residual is not None
        return summed, y

    @staticmethod
    def backward(ctx, dsum, dy):
        summed, weight = ctx.saved_tensors
        need_x, need_residual, need_weight, need_bias, _ = ctx.needs_input_grad
        if dy is None:
            return dsum, dsum.half() if need_residual and dsum is not None else None, None, None, None
        given = [dy] if dsum is None else [dy, dsum]
        if torch.is_grad_enabled() or not all(data_only(t) for t in given) or dy.dtype != torch.float16 \
                or (dsum is not None and dsum.dtype != torch.float32):
            # a graph of the gradients is wanted, or something follows them: operations that have one
            g = dy.float()
            h = summed - summed.mean(1, keepdim=True)
            rstd = (h.square().mean(1, keepdim=True) + ctx.eps).rsqrt()
            h, gw = h * rstd, g * weight
            dx = rstd * (gw - gw.mean(1, keepdim=True) - h * (gw * h).mean(1, keepdim=True))
            dx = dx if dsum is None else dx + dsum
            return (dx if need_x else None, dx.half() if need_residual else None, (g * h).sum(0) if need_weight else None,
                    g.sum(0) if need_bias else None, None)
        dy, dsum = (t if t is None or t.is_contiguous() and t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)
                    for t in (dy, dsum))
        (n, c), dev = summed.shape, summed.device
        dx = torch.empty_like(summed) if need_x else None
        dres = torch.empty_like(dy) if need_residual else None
        dgamma, dbeta = (torch.empty(c, dtype=torch.float32, device=dev) for _ in range(2))
        lib = _lib.lib()
        with _lib.on(dev):
            ws_bytes = lib.s3d_layernorm_grad_workspace_bytes(n, c)
            workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
            status = lib.s3d_layernorm_grad(
                summed.data_ptr(), None if dsum is None else dsum.data_ptr(), dy.data_ptr(), weight.data_ptr(), ctx.eps,
                None if dx is None else dx.data_ptr(), None if dres is None else dres.data_ptr(), dgamma.data_ptr(),
                dbeta.data_ptr(), n, c, workspace.data_ptr(), ws_bytes, _lib.stream(dev))
        _lib.check(status, "s3d_layernorm_grad")
        return dx, dres, dgamma if need_weight else None, dbeta if need_bias else None, None


def trained_add_norm(x, residual, norm):
    """(x + residual, norm(x + residual) in fp16) with gradients, for training under fp16 autocast where a dense layer takes
    the rows; None where it does not apply."""
    if followed() or not (torch.is_grad_enabled() and x.is_cuda and torch.is_autocast_enabled()
            and torch.get_autocast_dtype("cuda") == torch.float16 and plain(norm, nn.LayerNorm)):
        return None
    weight, bias = norm.weight, norm.bias
    if weight is None or bias is None or x.dim() != 2 or x.shape[0] == 0 or tuple(norm.normalized_shape) != (x.shape[1],) \
            or x.shape[1] % 4 or x.shape[1] > 1024:
        return None
    for t, dtype in ((x, torch.float32), (weight, torch.float32), (bias, torch.float32), (residual, torch.float16)):
        if t is not None and not (type(t) in (torch.Tensor, nn.Parameter) and t.dtype == dtype and t.device == x.device
                                  and t.is_contiguous() and t.data_ptr() % 16 == 0):
            return None
    if residual is not None and residual.shape != x.shape:
        return None
    return _AddNorm.apply(x, residual, weight, bias, norm)

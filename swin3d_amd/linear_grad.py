"""Dense layers in training under fp16 autocast, on the library's kernels: the forward on s3d_linear_in_order, the gradients on
s3d_linear (for the rows) and s3d_linear_grad (for weight and bias).  Tall rows and small weights are what the networks have,
where a product that does not split the sum over the rows leaves most of the chip idle.

The product of the forward is torch's to the bit, as it is outside of this file (has_torchs_bits has where it is made here).  A sum
over K in another order is no less exact, but it gives another sample of what fp16 activations do to the gradients of a network: on
scans of 5,000 to 40,000 voxels the gradients of Swin3D-S's encoder lie 1 to 5 % from those of an fp32 pass, and products that share
K among wavefronts in the forward moved them by 0.1 to 1.6 % (single elements by up to a seventh of the largest).  With torch's bits
they are what they were to the scatter of two runs, 0.05 to 0.1 %."""
import ctypes
import functools

import torch
import torch.nn.functional as F
from torch.autograd.function import Function

from . import _lib
from .swin_blocks import data_only, followed, linear_rows


_DTYPE_CODE = {torch.float32: _lib.S3D_DTYPE_F32, torch.float16: _lib.S3D_DTYPE_F16}


def _weight_gradients(dy, x, want_weight, want_bias, dtype=torch.float32):
    """(dy.T @ x, dy.sum(0)) of fp16 rows in `dtype`, as far as they are wanted; None where the kernel does not take them."""
    if not (data_only(dy) and data_only(x)) or dy.dtype != torch.float16 or dy.data_ptr() % 16 or x.data_ptr() % 16:
        return None
    if dy.shape[1] % 8:      # (the number of classes)
        extra = -dy.shape[1] % 8
        return tuple(g if g is None else g[:-extra].clone() for g in
                     _weight_gradients(F.pad(dy, (0, extra)), x, want_weight, want_bias, dtype))
    if x.shape[1] % 8:       # (the stem's 27 offsets)
        extra = -x.shape[1] % 8
        dw, db = _weight_gradients(dy, F.pad(x, (0, extra)), want_weight, want_bias, dtype)
        return dw if dw is None else dw[:, :-extra], db
    (m, n), k, dev = dy.shape, x.shape[1], dy.device
    dw = torch.empty((n, k), dtype=dtype, device=dev) if want_weight else None
    db = torch.empty(n, dtype=dtype, device=dev) if want_bias else None
    lib = _lib.lib()
    with _lib.on(dev):
        ws_bytes = lib.s3d_linear_grad_workspace_bytes(m, n, k)
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        status = lib.s3d_linear_grad(dy.data_ptr(), x.data_ptr(), None if dw is None else dw.data_ptr(),
                                     None if db is None else db.data_ptr(), _DTYPE_CODE[dtype], m, n, k, workspace.data_ptr(),
                                     ws_bytes, _lib.stream(dev))
    _lib.check(status, "s3d_linear_grad")
    return dw, db


# torch's library (hipBLASLt, of torch 2.10.0 for ROCm 7.0) adds up K in order, too, unless it splits it: for few rows or columns, for
# long K, and where a launch's last tiles would leave most of the chip idle.  Where it does not follows from results alone: of 1.28
# million products of random widths (N 8 to 2560, K 16 to 768) and 64 to 65,535 rows those inside the line are the same to the bit, and
# so are 126,000 of both networks' widths; outside of it lie 2,500 with N >= 32, none below 22.9 million numbers of a result, and 7,800
# with N = 8 to 24.  From 65,536 rows on 1 to 12 in 100 row counts have 10^-5 to 2 x 10^-4 of their numbers a rounding apart (K = 48 to
# N = 144: 67,301 rows), which moved the gradients of Swin3D-S by 0.3 to 0.6 % there; with torch's product 0.01 %, as two runs.
_LEAST_ROWS, _MANY_ROWS, _LEAST_N, _MOST_K = 64, 65536, 32, 768
_WIDE, _MOST_NUMBERS = 512, 20_000_000


def has_torchs_bits(m, n, k):
    """A product of m rows of k channels by a weight [n, k] in order is torch's."""
    return _LEAST_ROWS <= m < _MANY_ROWS and n >= _LEAST_N and k <= _MOST_K and (n < _WIDE or m * n <= _MOST_NUMBERS)


def dense_rows(x, weight, bias):
    """F.linear of fp16 operands in a forward that is trained: on the library's kernel where torch's has the same bits.  us, torch /
    so: 49,682 rows of 96 to 288 27 / 12, of 384 to 96 17 / 13; 12,421 of 192 to 576 16 / 9, of 768 to 192 10.2 / 10.3; 811 of 384 to
    384 5.3 / 4.6."""
    out = linear_rows(x, weight, bias, in_order=True) if x.dim() == 2 and has_torchs_bits(x.shape[0], *weight.shape) else None
    return F.linear(x, weight, bias) if out is None else out


@functools.lru_cache(maxsize=64)
def _copies_layout(rows, cols, with_bias, turned):
    """The copies that _half_copies makes, and where the weight's, its transpose and the bias's begin: on multiples of 512 bytes,
    as allocations of their own would."""
    step = rows * cols + -rows * cols % 256
    at = [0, step if turned else -1, step * (2 if turned else 1)]
    copies = (_lib.HalfCopy * 2)((rows, cols, 0, 0, at[1], -1, 1.0), (rows, 1, 0, at[2], -1, -1, 1.0))
    return copies, at, at[2] + (rows if with_bias else 0)


def _half_copies(weight, bias, turned):
    """(weight, its transpose or None, bias or None) in fp16 by one launch, in place of one each; None where they are not plain
    fp32 arrays of whole pieces."""
    given = [weight] if bias is None else [weight, bias]
    rows, cols = weight.shape
    if not weight.is_cuda or rows % 8 or cols % 8 or any(t.dtype != torch.float32 or not t.is_contiguous() or t.data_ptr() % 16 for t in given):
        return None
    copies, at, count = _copies_layout(rows, cols, bias is not None, turned)
    half = torch.empty(count, dtype=torch.float16, device=weight.device)
    with _lib.on(weight.device):
        status = _lib.lib().s3d_half_copies((ctypes.c_void_p * len(given))(*[t.data_ptr() for t in given]), copies, len(given), half.data_ptr(), None,
                                            _lib.stream(weight.device))
    _lib.check(status, "s3d_half_copies")
    return (half.as_strided((rows, cols), (cols, 1), 0), half.as_strided((cols, rows), (rows, 1), at[1]) if turned else None,
            None if bias is None else half.as_strided((rows,), (1,), at[2]))


class _Linear(Function):
    """F.linear in fp16 of fp16 rows and parameters in fp16 or fp32, whose gradients come in their own type: autocast would
    round them to fp16 on the way."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        copies = _half_copies(weight, bias, ctx.needs_input_grad[0])
        half, turned, half_bias = copies if copies is not None else (
            weight.to(torch.float16), None, None if bias is None else bias.to(torch.float16))
        ctx.save_for_backward(x, weight, half, turned)
        ctx.bias_dtype = None if bias is None else bias.dtype
        return dense_rows(x, half, half_bias)

    @staticmethod
    def backward(ctx, dy):
        x, weight, half, turned = ctx.saved_tensors
        need_x, need_weight, need_bias = ctx.needs_input_grad
        dx = grads = None
        if not torch.is_grad_enabled():
            dy = dy.contiguous()
            if need_x:
                dx = linear_rows(dy, half.t().contiguous() if turned is None else turned, None)
                dx = dy.mm(half) if dx is None else dx
            if need_weight or need_bias:
                grads = _weight_gradients(dy, x.contiguous(), need_weight, need_bias, weight.dtype if need_weight else ctx.bias_dtype)
        elif need_x:      # a graph of the gradients is wanted: operations that have one
            dx = dy.mm(weight.to(torch.float16))
        if grads is None:
            grads = dy.t().mm(x) if need_weight else None, dy.sum(0) if need_bias else None
        dw, db = grads
        return dx, dw if dw is None else dw.to(weight.dtype), db if db is None else db.to(ctx.bias_dtype)


def trained_linear(x, weight, bias, any_width=False):
    """F.linear(x, weight, bias) as autocast computes it, with the gradients above; None where this does not apply: outside
    of training under fp16 autocast, and for operands that the kernels do not take.  any_width: also rows of no whole number
    of 16-byte pieces, which the weight's gradient then copies."""
    if not (torch.is_grad_enabled() and x.is_cuda and torch.is_autocast_enabled()
            and torch.get_autocast_dtype("cuda") == torch.float16):
        return None
    for t in (x, weight, bias):
        if t is not None and (type(t) not in (torch.Tensor, torch.nn.Parameter) or t.device != x.device
                              or t.dtype not in (torch.float16, torch.float32)):
            return None
    if x.dim() != 2 or weight.dim() != 2 or x.shape[0] == 0 or x.shape[1] != weight.shape[1] or (x.shape[1] % 8 and not any_width) \
            or x.shape[1] == 0 or weight.shape[0] == 0 or max(weight.shape) > 16384 \
            or (bias is not None and bias.shape != weight.shape[:1]) or followed():
        return None
    return _Linear.apply(x.to(torch.float16), weight, bias)

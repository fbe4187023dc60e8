"""ctypes loader of libswin3d_amd.so (the C-ABI HIP library declared in include/swin3d_amd.h).

There is no fallback: if the shared library is missing or a call fails, a
RuntimeError is raised.
"""
import contextlib
import ctypes
import os

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libswin3d_amd.so")

S3D_DTYPE_F32 = 0
S3D_DTYPE_F16 = 1
S3D_DTYPE_F32_F16_ROWS = 2     # s3d_attn_bwd only: fp32 tables beside fp16 rows
KNN_KMAX = 64
S3D_ATTN_PLANNED = 4
S3D_ATTN_SIZES_ON_DEVICE = 8

_lib = None

_vp = ctypes.c_void_p
_i32 = ctypes.c_int32
_i64 = ctypes.c_int64


class WindowSet(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("w_sizes", "w2n", "n2n", "n_coords")] + [
        ("num_windows", _i64), ("plan", _vp), ("plan_bytes", ctypes.c_size_t), ("planned", _i32)]


class WindowIndexSet(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("n2n", "w_w_id", "w_sizes", "w2n", "counts")] + [("window", _i32), ("shift", _i32)]


class SwinBlock(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("norm1_weight", "norm1_bias", "norm2_weight", "norm2_bias", "qkv_weight", "qkv_bias",
                                   "table_q", "table_k", "table_v", "proj_weight", "proj_bias", "fc1_weight", "fc1_bias",
                                   "fc2_weight", "fc2_bias")] + [("norm1_eps", ctypes.c_float), ("norm2_eps", ctypes.c_float)]


class HalfCopy(ctypes.Structure):
    _fields_ = [(n, _i64) for n in ("rows", "cols", "scaled_rows", "to", "transposed", "same")] + [("scale", ctypes.c_float)]


class BlockPass(ctypes.Structure):
    _fields_ = [("params", ctypes.POINTER(_vp)), ("copies", ctypes.POINTER(HalfCopy)), ("num_copies", _i64), ("half", _vp), ("same", _vp),
                *((n, _i64) for n in ("qkv_weight", "qkv_bias", "proj_weight", "proj_bias", "fc1_weight", "fc1_bias", "fc2_weight", "fc2_bias",
                                      "table_q", "table_k", "table_v")),
                *((n, _vp) for n in ("norm2_weight", "norm2_bias", "x", "normed1", "qkv", "attended", "out_max", "out_sum", "sum", "normed2",
                                     "hidden_in", "hidden_out", "pending")),
                ("windows", ctypes.POINTER(WindowSet)), ("norm2_eps", ctypes.c_float)]


class BlockSaved(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("normed1", "qkv", "attended", "out_max", "out_sum", "sum", "normed2", "hidden_in", "hidden_out",
                                   "qkv_weight_t", "proj_weight_t", "fc1_weight_t", "fc2_weight_t", "table_q", "table_k", "table_v",
                                   "norm2_weight", "w_sizes", "w2n", "n2n", "n_coords")] + [("norm2_eps", ctypes.c_float)]


class BlockGradients(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("x", "normed1", "norm2_weight", "norm2_bias", "qkv_weight", "qkv_bias", "proj_weight", "proj_bias",
                                   "fc1_weight", "fc1_bias", "fc2_weight", "fc2_bias", "table_q", "table_k", "table_v")]


# name -> (restype, argtypes); mirrors include/swin3d_amd.h
SIGNATURES = {
    "s3d_version": (ctypes.c_int, []),
    "s3d_last_error_string": (ctypes.c_char_p, []),
    "s3d_attn_fwd_workspace_bytes": (ctypes.c_size_t, [_i32, _i64, _i64]),
    "s3d_attn_fwd": (ctypes.c_int, [_vp] * 7 + [_i32, _i64] + [_vp] * 7 +
                     [_i64, _i32, _i32, _i64, _i64, _i32, _i32, _vp, ctypes.c_size_t, _vp]),
    "s3d_attn_plan_bytes": (ctypes.c_size_t, [_i32, _i64, _i64]),
    "s3d_attn_plan": (ctypes.c_int, [_vp, _i32, _i64, _vp, _vp, _i64, _i32, _i32, _i64, _i32, _vp, ctypes.c_size_t, _vp]),
    "s3d_attn_fwd_noalloc": (ctypes.c_int, [_vp] * 7 + [_i32, _i64] + [_vp] * 7 +
                             [_i64, _i32, _i32, _i64, _i64, _i32, _vp]),
    "s3d_attn_bwd_workspace_bytes": (ctypes.c_size_t, [_i32, _i32, _i32, _i64, _i64, _i64, _i64]),
    "s3d_attn_bwd_workspace_least_bytes": (ctypes.c_size_t, [_i32, _i32, _i32, _i64, _i64, _i64, _i64]),
    # q k v tq tk tv sizes | nd len | w_sizes w2n n2n coords out max sum dout dq dk dv dtq dtk dtv | N H D W pairs dtype | ws bytes stream
    "s3d_attn_bwd": (ctypes.c_int, [_vp] * 7 + [_i32, _i64] + [_vp] * 14 +
                     [_i64, _i32, _i32, _i64, _i64, _i32, _vp, ctypes.c_size_t, _vp]),
    # ... pairs, row strides of q, k, v and of dq, dk, dv, dtype ...
    "s3d_attn_bwd_strided": (ctypes.c_int, [_vp] * 7 + [_i32, _i64] + [_vp] * 14 +
                             [_i64, _i32, _i32, _i64, _i64, _i64, _i64, _i32, _vp, ctypes.c_size_t, _vp]),
    "s3d_window_index_workspace_bytes": (ctypes.c_size_t, [_i64]),
    "s3d_window_index": (ctypes.c_int, [_vp, _i64, _i32, _i32, _i32] + [_vp] * 6 + [ctypes.c_size_t, _vp]),
    "s3d_gather_rows": (ctypes.c_int, [_vp, _i64, _vp, _i64, _i32, _i32, _vp, _vp]),
    "s3d_voxel_neighbours_workspace_bytes": (ctypes.c_size_t, [_i64]),
    "s3d_voxel_neighbours": (ctypes.c_int, [_vp, _i64, _i32, _i32, _vp, _vp, ctypes.c_size_t, _vp]),
    "s3d_segment_ends": (ctypes.c_int, [_vp, _i64, _i64, _i32, _vp, _vp]),
    "s3d_segment_ends_of_two": (ctypes.c_int, [_vp, _i64, _i64, _vp, _i64, _i64, _i32, _vp, _vp]),
    "s3d_pool_cells": (ctypes.c_int, [_vp, _vp, _vp, _i64, _vp, _i32, _vp, _i64, _i32, _vp, _vp, _vp, _vp]),
    "s3d_level_signals": (ctypes.c_int, [_vp, _vp, _vp, _i32, _vp, _i64, _i32, _i32, ctypes.c_float, ctypes.c_float, _vp, _i64, _vp]),
    "s3d_knn_strided": (ctypes.c_int, [_i32, _vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i32, _vp, _vp, ctypes.c_float, _vp,
                                       ctypes.c_size_t, _vp]),
    "s3d_half_copies": (ctypes.c_int, [_vp, _vp, _i32, _vp, _vp, _vp]),
    "s3d_add_half": (ctypes.c_int, [_vp, _vp, _vp, _i64, _vp]),
    "s3d_swin_block_grad_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32, _i32, _i32, _i64, _i64, _i64]),
    # saved grads dsum dpending | N H D hidden | sizes nd len | W pairs scale dtype | ws bytes stream
    "s3d_stem_workspace_bytes": (ctypes.c_size_t, [_i64, _i32]),
    "s3d_stem": (ctypes.c_int, [_vp, _i32, _i64, _i32, _vp, _vp, _i32] + [_vp] * 4 + [ctypes.c_float, _vp, _vp, ctypes.c_size_t, _vp]),
    "s3d_swin_block_train": (ctypes.c_int, [_vp, _i64, _i32, _i32, _i32, _vp, _i32, _i64, _vp]),
    "s3d_swin_block_grad": (ctypes.c_int, [_vp] * 4 + [_i64, _i32, _i32, _i32, _vp, _i32, _i64, _i64, _i64, ctypes.c_float, _i32, _vp,
                                           ctypes.c_size_t, _vp]),
    "s3d_cast_half": (ctypes.c_int, [_vp, _vp, _vp, _i32, _vp]),
    "s3d_window_index_grid_workspace_bytes": (ctypes.c_size_t, [_i64]),
    "s3d_window_index_grid": (ctypes.c_int, [_vp, _i64, _i32, _i32, _i32] + [_vp] * 6 + [ctypes.c_size_t, _vp]),
    "s3d_window_indices_workspace_bytes": (ctypes.c_size_t, [_i64, _i32]),
    "s3d_window_indices": (ctypes.c_int, [_vp, _i64, _i32, _vp, _i32, _vp, ctypes.c_size_t, _vp]),
    "s3d_window_indices_counted": (ctypes.c_int, [_vp, _i64, _i32, _vp, _i32, _vp, _vp, ctypes.c_size_t, _vp]),
    "s3d_window_indices_finished": (ctypes.c_int, [_vp, _i64, _i32, _vp, _i32, _vp, _vp, ctypes.c_size_t, _vp]),
    "s3d_cell_representatives": (ctypes.c_int, [_vp, _vp, _vp, _i64, _vp, _i64, _i32, _vp, _vp]),
    "s3d_key_neighbours": (ctypes.c_int, [_vp, _vp, _i64, _vp, _i32, _vp, _vp]),
    "s3d_window_signals": (ctypes.c_int, [_vp, _vp, _vp, _vp, _i64, _i32, _i32, ctypes.c_float, ctypes.c_float, _vp,
                                          _i64, _vp]),
    "s3d_knn_workspace_bytes": (ctypes.c_size_t, [_i64, _i64, _i32]),
    "s3d_knn": (ctypes.c_int, [_i32, _vp, _i64, _vp, _i64, _vp, _vp, _i32, _vp, _vp, ctypes.c_float,
                               _vp, ctypes.c_size_t, _vp]),
    "s3d_knn_distances": (ctypes.c_int, [_i32, _vp, _i64, _vp, _i64, _vp, _vp, _i32, _vp, _vp, ctypes.c_float,
                               _vp, ctypes.c_size_t, _vp]),
    "s3d_knn_interpolate_add": (ctypes.c_int, [_vp, _vp, _i32, _i64, _vp, _i64, _i32, _vp, _vp, _vp]),
    "s3d_knn_interpolate_grad": (ctypes.c_int, [_vp, _vp, _i32, _i64, _vp, _i64, _i32, _vp, _vp, _vp]),
    "s3d_knn_interpolate": (ctypes.c_int, [_vp, _vp, _i32, _i64, _vp, _i64, _i32, _i32, _vp, _vp]),
    "s3d_knn_max_pool": (ctypes.c_int, [_vp, _i32, _i64, _vp, _i64, _i32, _i32, _vp, _vp]),
    "s3d_knn_max_pool_widened": (ctypes.c_int, [_vp, _i32, _i64, _vp, _i64, _i32, _vp, _vp]),
    "s3d_knn_max_pool_grad_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i64, _i32, _i32]),
    "s3d_knn_max_pool_grad": (ctypes.c_int, [_vp, _i32, _i64, _vp, _i64, _i32, _i32, _vp, _vp, _vp, _vp, ctypes.c_size_t, _vp]),
    "s3d_add_layernorm": (ctypes.c_int, [_vp, _vp, _i32, _vp, _vp, ctypes.c_float, _vp, _vp, _i32, _i64, _i32, _vp]),
    "s3d_train_add_layernorm": (ctypes.c_int, [_vp] * 4 + [ctypes.c_float, _vp, _vp, _i64, _i32, _vp]),
    "s3d_layernorm_grad_workspace_bytes": (ctypes.c_size_t, [_i64, _i32]),
    "s3d_layernorm_grad": (ctypes.c_int, [_vp] * 4 + [ctypes.c_float] + [_vp] * 4 + [_i64, _i32, _vp, ctypes.c_size_t, _vp]),
    "s3d_linear": (ctypes.c_int, [_vp] * 4 + [_i64, _i32, _i32, _i32, _vp]),
    "s3d_linear_in_order": (ctypes.c_int, [_vp] * 5 + [_i64, _i32, _i32, _vp]),
    "s3d_mlp": (ctypes.c_int, [_vp] * 6 + [_i64, _i32, _i32, _vp]),
    "s3d_linear_grad_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32]),
    "s3d_linear_grad": (ctypes.c_int, [_vp] * 4 + [_i32, _i64, _i32, _i32, _vp, ctypes.c_size_t, _vp]),
    "s3d_swin_blocks_workspace_bytes": (ctypes.c_size_t, [_i64, _i32, _i32]),
    # x x_out pending | N H D hidden | table sizes nd len | sets blocks | ws bytes stream
    "s3d_swin_blocks": (ctypes.c_int, [_vp] * 3 + [_i64, _i32, _i32, _i32] + [_vp, _i32, _i64] + [_vp, _i32] * 2 +
                        [_vp, ctypes.c_size_t, _vp]),
}


def lib():
    """The loaded library; raises RuntimeError when it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `python -m swin3d_amd.build` "
                "(hipcc --offload-arch=gfx950); swin3d_amd has no CPU or PyTorch fallback")
        handle = ctypes.CDLL(LIB_PATH)
        for name, (restype, argtypes) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = restype
            fn.argtypes = argtypes
        _lib = handle
    return _lib


_HERE_ALREADY = contextlib.nullcontext()


def on(device):
    """Context with `device` (that of a CUDA tensor) as the current one; nothing to do where it is so already, which is
    a tenth of what torch.cuda.device costs the host."""
    return _HERE_ALREADY if torch.cuda.current_device() == device.index else torch.cuda.device(device)


def stream(device):
    """The current stream of `device` as the library takes it."""
    return torch._C._cuda_getCurrentRawStream(device.index)


def cast_half(tensors):
    """fp32 CUDA tensors (of one device) in fp16, flat copies in one launch: [tensor of the same shape, contiguous]."""
    done = []
    for first in range(0, len(tensors), 16):
        some = [t.contiguous() for t in tensors[first:first + 16]]
        out = [torch.empty(t.shape, dtype=torch.float16, device=t.device) for t in some]
        num = len(some)
        sources, targets, counts = (ctypes.c_void_p * num)(), (ctypes.c_void_p * num)(), (ctypes.c_int64 * num)()
        for i, (t, o) in enumerate(zip(some, out)):
            sources[i], targets[i], counts[i] = t.data_ptr(), o.data_ptr(), t.numel()
        with on(some[0].device):
            status = lib().s3d_cast_half(sources, targets, counts, num, stream(some[0].device))
        check(status, "s3d_cast_half")
        done += out
    return done


def check(status, what):
    if status != 0:
        msg = lib().s3d_last_error_string().decode("utf-8", "replace")
        kind = ValueError if status < 0 else RuntimeError
        raise kind(f"{what} failed with status {status}: {msg}")

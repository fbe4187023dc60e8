"""The Swin blocks of a stage at inference under fp16 autocast as one library call (s3d_swin_blocks): the host's share of
a block through torch is some fifteen dispatches, several times what its kernels take on a small scan."""
import ctypes

import torch
import torch.nn as nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _module_hooks

from . import _lib
from .sparse_dl.attn import attn_coff


def plain(m, kind):
    """m is a `kind` (no subclass: it may compute something else) and nothing watches or replaces its forward."""
    return (type(m) is kind and not m._forward_hooks and not m._forward_pre_hooks and "forward" not in m.__dict__
            and not m._backward_hooks and not m._backward_pre_hooks
            and not _module_hooks._global_forward_hooks and not _module_hooks._global_forward_pre_hooks
            and not _module_hooks._global_backward_hooks and not _module_hooks._global_backward_pre_hooks)


def followed():
    """Something follows what is done to tensors, which a call by address would pass by: a transform, a forward-mode
    derivative, a dispatch mode or a tracer."""
    return (forward_ad._current_level >= 0 or torch._C._functorch.peek_interpreter_stack() is not None
            or torch._C._len_torch_dispatch_stack() > 0 or torch.jit.is_tracing() or torch.compiler.is_compiling())


def data_only(x):
    """x is its data (no subclass) and nothing follows what is done to it."""
    return type(x) is torch.Tensor and not followed()


def _parts(block, kinds):
    """(block, norm1, attn, qkv, proj, norm2, mlp, fc1, act, fc2), or None where one of them is not what it was built as."""
    m = block._modules
    attn, mlp = m["attn"], m["mlp"]
    if not (plain(block, kinds[0]) and plain(attn, kinds[1]) and plain(mlp, kinds[2])):
        return None
    a, f = attn._modules, mlp._modules
    parts = (block, m["norm1"], attn, a["qkv"], a["proj"], m["norm2"], mlp, f["fc1"], f["act"], f["fc2"])
    if not (plain(parts[1], nn.LayerNorm) and plain(parts[5], nn.LayerNorm) and plain(parts[8], nn.GELU)
            and parts[8].approximate == "none" and all(plain(parts[i], nn.Linear) for i in (3, 4, 7, 9))):
        return None
    return parts


def _stamp(parts):
    """What the descriptions of the blocks, and the decision that there are any, follow from: addresses and versions of the
    parameters, and the plain attributes of the layers, which a program may set at any time."""
    stamp = [x for block in parts for i in (1, 2, 3, 4, 5, 7, 9) for p in block[i]._parameters.values() if p is not None
             for x in (p.data_ptr(), p._version)]
    for _, norm1, attn, qkv, proj, norm2, _, fc1, _, fc2 in parts:
        stamp += [attn.fp16_mode, attn.num_heads, attn.head_dim, attn.dim, attn.scale, attn.cRSE, *attn.table_sizes]
        stamp += [x for norm in (norm1, norm2) for x in (norm.eps, *norm.normalized_shape)]
        stamp += [x for layer in (qkv, proj, fc1, fc2) for x in (layer.in_features, layer.out_features)]
    return stamp


class _Kept:
    """What swin_blocks keeps on its owner: key, descriptions (or None) and the tensors they point to.  Addresses are
    worth nothing in another place: a copy of the owner, or one read from a file, starts with None."""

    def __init__(self, key, described, tensors):
        self.key, self.described, self.tensors = key, described, tensors

    def __reduce__(self):
        return type(None), ()


def _descriptions(parts, half_copy):
    """The blocks as the library takes them, and the tensors they point to.  half_copy: (layer) -> its (weight, bias) in
    fp16, for parameters that are not copied by one launch."""
    from .swin_train import packed_copies      # (which reads this module)
    kept, blocks = [], (_lib.SwinBlock * len(parts))()

    def at(t):
        if t is None:
            return None
        kept.append(t)
        return t.data_ptr()

    for b, block in zip(blocks, parts):
        _, norm1, attn, _, proj, norm2, _, fc1, _, fc2 = block
        packed = packed_copies(block)
        if packed is not None:
            kept.append(packed[0])
            (b.qkv_weight, b.qkv_bias, b.proj_weight, b.proj_bias, b.fc1_weight, b.fc1_bias, b.fc2_weight, b.fc2_bias,
             b.table_q, b.table_k, b.table_v) = packed[1]
        else:
            weight, bias, tables = attn._prepared()
            b.qkv_weight, b.qkv_bias = at(weight.contiguous()), at(bias)
            b.table_q, b.table_k, b.table_v = (at(t) for t in tables)
            for name, layer in (("proj", proj), ("fc1", fc1), ("fc2", fc2)):
                w, bias = half_copy(layer)
                setattr(b, name + "_weight", at(w.contiguous()))
                setattr(b, name + "_bias", at(bias))
        for name, norm in (("norm1", norm1), ("norm2", norm2)):
            setattr(b, name + "_weight", at(norm.weight.detach().float().contiguous()))
            setattr(b, name + "_bias", at(norm.bias.detach().float().contiguous()))
            setattr(b, name + "_eps", norm.eps)
    return blocks, kept


def _applicable(parts, channels):
    attn, fc1 = parts[0][2], parts[0][7]
    if attn.fp16_mode not in (1, 2) or attn.head_dim not in (8, 16, 32) or channels % 16 or fc1.out_features % 16:
        return False
    for _, norm1, a, qkv, proj, norm2, _, f1, _, f2 in parts:
        if (a.num_heads, a.head_dim, a.fp16_mode, a.dim) != (attn.num_heads, attn.head_dim, attn.fp16_mode, channels) \
                or list(a.table_sizes) != list(attn.table_sizes):
            return False
        for norm in (norm1, norm2):
            if tuple(norm.normalized_shape) != (channels,) or norm.weight is None or norm.bias is None:
                return False
        shapes = [(qkv, channels, 3 * channels), (proj, channels, channels), (f1, channels, fc1.out_features),
                  (f2, fc1.out_features, channels)]
        if any((m.in_features, m.out_features) != (i, o) for m, i, o in shapes):
            return False
        # the fp16 copies of fp32 parameters on one device
        if any(p.dtype != torch.float32 or p.device != qkv.weight.device
               for m in (norm1, a, qkv, proj, norm2, f1, f2) for p in m._parameters.values() if p is not None):
            return False
    return True


def linear_rows(x, weight, bias, gelu=False, in_order=False):
    """x @ weight.T + bias (then GELU) of fp16 rows on the library's kernel (s3d_linear; in_order: without GELU, on
    s3d_linear_in_order); None where it does not take the operands."""
    if not data_only(x) or x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1] \
            or any(t is not None and (t.dtype != torch.float16 or t.device != x.device or not t.is_contiguous()
                                      or t.data_ptr() % 16) for t in (x, weight, bias)) \
            or x.shape[1] % 16 or x.shape[1] == 0 or weight.shape[0] % 8 or weight.shape[0] == 0 \
            or (bias is not None and bias.shape != weight.shape[:1]):
        return None
    out = torch.empty((x.shape[0], weight.shape[0]), dtype=torch.float16, device=x.device)
    with _lib.on(x.device):
        operands = x.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), out.data_ptr()
        sizes, stream = (x.shape[0], weight.shape[0], x.shape[1]), _lib.stream(x.device)
        status = _lib.lib().s3d_linear_in_order(*operands, None, *sizes, stream) if in_order else \
            _lib.lib().s3d_linear(*operands, *sizes, int(gelu), stream)
    _lib.check(status, "s3d_linear")
    return out


def swin_blocks(owner, blocks, kinds, feats, index_sets, epoch, half_copy):
    """(feats, pending) behind the blocks, as their `forward_fused` one after the other would give it, or None where the
    library call does not stand for them.

    owner       the module that keeps the descriptions of the blocks between calls (`_s3d_blocks`), made anew when a
                parameter, its version, an attribute of a layer or `epoch` has changed
    kinds       (block, attention, MLP) types the blocks have to be of
    feats       fp32 [N,C]; left as it is
    index_sets  per window set what index_arguments and window_signals give
    """
    n, channels = feats.shape
    if n == 0 or not data_only(feats) or any(len(s) < 9 for s in index_sets):
        return None
    parts = [_parts(b, kinds) for b in blocks]
    if any(p is None for p in parts):
        return None
    key = (epoch, _stamp(parts), [m for p in parts for m in p])
    kept = getattr(owner, "_s3d_blocks", None)
    if kept is None or kept.key != key:
        kept = _Kept(key, *(_descriptions(parts, half_copy) if _applicable(parts, channels) else (None, None)))
        owner._s3d_blocks = kept
    if kept.described is None:
        return None
    described, tensors = kept.described, kept.tensors
    dev = feats.device
    if tensors[0].device != dev:
        return None
    attn, hidden = parts[0][2], parts[0][7].out_features
    heads, dim, sizes = attn.num_heads, attn.head_dim, attn.table_sizes
    nd, table_len = len(sizes), sum(sizes)
    c_sizes = (ctypes.c_int32 * nd)(*sizes)
    lib = _lib.lib()
    feats = feats.contiguous()
    out = torch.empty_like(feats)
    pending = torch.empty((n, channels), dtype=torch.float16, device=dev)
    ws_bytes = lib.s3d_swin_blocks_workspace_bytes(n, channels, hidden)
    workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    sets = (_lib.WindowSet * len(index_sets))()
    held = []
    with _lib.on(dev):
        stream = _lib.stream(dev)
        for s, args in zip(sets, index_sets):
            w_sizes_in, w2n_in, n2n, coords = args[3], args[4], args[5], args[8]
            w_sizes, w2n = (attn_coff._as_int32(name, t, dev) for name, t in (("w_sizes", w_sizes_in), ("w2n", w2n_in)))
            n2n = None if n2n is None else attn_coff._as_int32("n2n", n2n, dev)
            coords = coords.float().contiguous()
            if w_sizes.dim() != 1 or w2n.shape != w_sizes.shape or coords.shape != (n, nd) or coords.device != dev \
                    or (n2n is not None and n2n.shape != (n,)):
                return None
            plan = attn_coff._plan_for(lib, w_sizes_in, w2n_in, w_sizes, w2n, c_sizes, sizes, nd, table_len, n, heads, dim,
                                       _lib.S3D_DTYPE_F16, stream) if attn_coff.REUSE_PLANS else None
            s.planned = plan is not None
            if plan is None:
                plan = torch.empty(lib.s3d_attn_plan_bytes(heads, n, w_sizes.numel()), dtype=torch.uint8, device=dev)
            held.append((w_sizes, w2n, n2n, coords, plan))
            s.w_sizes, s.w2n, s.n_coords = w_sizes.data_ptr(), w2n.data_ptr(), coords.data_ptr()
            s.n2n = None if n2n is None else n2n.data_ptr()
            s.num_windows, s.plan, s.plan_bytes = w_sizes.numel(), plan.data_ptr(), plan.numel()
        status = lib.s3d_swin_blocks(
            feats.data_ptr(), out.data_ptr(), pending.data_ptr(), n, heads, dim, hidden, c_sizes, nd, table_len, sets,
            len(sets), described, len(described), workspace.data_ptr(), ws_bytes, stream)
    _lib.check(status, "s3d_swin_blocks")
    return out, pending

"""A Swin block behind its first LayerNorm in training under fp16 autocast, as one node of autograd:

    sum = x + proj(attention(qkv(normed)));  pending = fc2(GELU(fc1(LayerNorm(sum))))

Layer by layer that is a dozen nodes, some thirty copies and casts of parameters and fifty dispatches of the backward, which
on scans of up to 100,000 voxels take the host longer than the kernels take the device.  Here the parameters are cast,
scaled and transposed by one launch (s3d_half_copies), and forward and backward are one call of the library each
(s3d_swin_block_train, s3d_swin_block_grad).

The forward's products and norm are torch's to the bit, as in linear_grad.py, for the reason given there."""
import ctypes
import functools
import itertools

import torch
import torch.nn.functional as F
from torch.autograd.function import Function

from . import _lib
from .fused_norm import _AddNorm, train_add_layernorm
from .linear_grad import _Linear, dense_rows, has_torchs_bits
from .sparse_dl.attn import attn_coff
from .sparse_dl.attn.attn_coff import IndexMode, PosEmb, PrecisionMode, SelfAttnAIOFunction, TableDims
from .swin_blocks import _applicable, _parts, data_only, followed

_PRECISION = (PrecisionMode.HALF_NONE, PrecisionMode.HALF_FORWARD, PrecisionMode.HALF_ALL)
_KINDS = ("query", "key", "value")
_GROUPS = ("xyz", "rgb", "norm")


class _Layout:
    """Where the fp16 copies of a block's parameters lie in one buffer, by the shapes alone: per array (rows, columns) of
    `shapes`, in the order of _parameters.  Every copy of a layer starts on a multiple of 512 bytes, as an allocation of
    its own would: the library behind torch's products picks kernels by alignment.  turned: with transposed copies of the
    weights, which a backward reads."""

    def __init__(self, shapes, num_tables, scaled_rows, scale, same_tables, turned=True):
        layers = len(shapes) - num_tables
        self.copies = (_lib.HalfCopy * len(shapes))()
        self.shapes, self.to, self.transposed = shapes, [], []
        at = same = 0
        for i, (copy, (rows, cols)) in enumerate(zip(self.copies, shapes)):
            table = i >= layers
            # (a kind's tables lie one behind the other, as the attention reads them)
            at += 0 if table and (i - layers) % (num_tables // 3) else -at % 256
            across = turned and not table and cols > 1
            copy.rows, copy.cols, copy.to = rows, cols, at
            at += rows * cols
            if across:
                at += -at % 256
            copy.transposed = at if across else -1
            at += rows * cols if across else 0
            copy.scaled_rows, copy.scale = (scaled_rows, scale) if rows == 3 * scaled_rows and i < 2 else (0, 1.0)
            copy.same = same if table and same_tables else -1
            same += rows * cols if table and same_tables else 0
            self.to.append(copy.to)
            self.transposed.append(copy.transposed)
        self.half_count, self.same_count = at, same


_layout = functools.lru_cache(maxsize=64)(_Layout)


def _shapes(params):
    return tuple((p.shape[0], p.shape[1]) if p.dim() == 2 else (p.numel(), 1) for p in params)


def packed_copies(parts):
    """What inference reads of a block's parameters, in fp16 and with the scale of q in, by one launch: the buffer that has
    them and [address or None of qkv weight, bias, proj .., fc1 .., fc2 .., query, key, value tables] in it; None where they
    are not plain fp32 arrays.  `parts` has passed _applicable."""
    attn = parts[2]
    groups = len(attn.table_sizes) // 3
    params = _parameters(parts, groups)
    dev = params[0].device
    if type(attn.scale) is not float or not params[0].is_cuda or followed() or any(t is None for t in params[8:]) \
            or any(t is not None and not (type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_contiguous()) for t in params):
        return None
    given = [p for p in params if p is not None]
    layout = _layout(_shapes(given), 3 * groups, attn.dim, attn.scale, False, False)
    half = torch.empty(layout.half_count, dtype=torch.float16, device=dev)
    with _lib.on(dev):
        status = _lib.lib().s3d_half_copies((ctypes.c_void_p * len(given))(*[p.data_ptr() for p in given]), layout.copies, len(given),
                                            half.data_ptr(), None, _lib.stream(dev))
    _lib.check(status, "s3d_half_copies")
    base, places = half.data_ptr(), iter(layout.to)
    layers = [None if p is None else base + 2 * next(places) for p in params[:8]]
    return half, layers + [base + 2 * at for at in layout.to[-3 * groups::groups]]


class _Call:
    """What a block's pass needs besides tensors that have gradients."""
    __slots__ = ("heads", "dim", "hidden", "sizes", "table_len", "index", "mode", "eps", "scale", "pairs")


def _parameters(parts, groups):
    """[qkv weight, bias, proj .., fc1 .., fc2 .., query tables, key tables, value tables] of a block; biases may be None."""
    _, _, attn, qkv, proj, _, _, fc1, _, fc2 = parts
    tables = attn._parameters
    return [p for layer in (qkv, proj, fc1, fc2) for p in (layer.weight, layer.bias)] + [
        tables.get(f"{kind}_{name}_table") for kind in _KINDS for name in _GROUPS[:groups]]


_CHECKED = (2, 4, 6)       # of _parameters: the weights of proj, fc1 and fc2


def _unchecked(norm_bias, params):
    """The parameters that a program may change in place between forward and backward, as it may with the nodes of the
    single layers: those leave a weight or a norm's input for the backward, but no bias, and of q, k, v's weight and of the
    tables a product or a copy."""
    return [norm_bias, *(p for i, p in enumerate(params) if i not in _CHECKED)]


def trained_branches(block, kinds, x, normed, attn_args):
    """(sum, pending) of `block` (of the types `kinds`) for rows x and their first norm `normed`, which trained_add_norm
    made; None where the layers have to be called one by one."""
    n, channels = x.shape
    parts = _parts(block, kinds)
    if parts is None or len(attn_args) < 9 or normed.dtype != torch.float16 or not _applicable([parts], channels) or followed() \
            or type(parts[2].scale) is not float:
        return None
    _, _, attn, _, _, norm2, _, fc1, _, _ = parts
    sizes, heads, dim, dev = list(attn.table_sizes), attn.num_heads, attn.head_dim, x.device
    nd, table_len = len(sizes), sum(sizes)
    params = _parameters(parts, nd // 3)
    for t in (norm2.weight, norm2.bias, *params):
        if t is not None and not (type(t) in (torch.Tensor, torch.nn.Parameter) and t.dtype == torch.float32 and t.device == dev
                                  and t.is_contiguous() and t.data_ptr() % 16 == 0):
            return None
    tables = params[8:]
    w_sizes, w2n, n2n, coords = attn_args[3], attn_args[4], attn_args[5], attn_args[8]
    per_kind = nd // 3
    if nd not in (3, 6, 9) or heads * dim != channels or dim == 32 or table_len > attn_coff.BWD_MAX_ROWS_PER_AXIS * nd * channels \
            or any(t is None for t in tables) or any(t.numel() != sum(sizes[3 * (i % per_kind):3 * (i % per_kind) + 3]) for i, t in enumerate(tables)) \
            or not (data_only(coords) and coords.dtype == torch.float32 and coords.shape == (n, nd) and coords.is_contiguous()
                    and coords.device == dev) \
            or any(not (data_only(t) and t.device == dev and t.dtype in (torch.int32, torch.int64)) for t in (w_sizes, w2n)) \
            or not (n2n is None or data_only(n2n) and n2n.device == dev and n2n.dtype in (torch.int32, torch.int64)):
        return None
    # (a replay gives a gradient to the tensors themselves, whatever became of them since the forward: they have to be leaves)
    if any(t is not None and t.grad_fn is not None for t in _unchecked(norm2.bias, params)):
        return None
    # (a pass that leaves nothing for the attention's backward runs other kernels)
    if not (normed.requires_grad or any(t.requires_grad for t in itertools.chain(params[:2], tables) if t is not None)):
        return None
    pairs = attn_coff._pairs_of(w_sizes, w_sizes) if attn_coff.BWD_PAIR_STORE else 0
    if pairs == 0 or not attn_coff._pair_store_fits(pairs, heads):
        return None
    call = _Call()
    call.heads, call.dim, call.hidden, call.sizes, call.table_len = heads, dim, fc1.out_features, sizes, table_len
    call.index, call.mode, call.eps, call.scale, call.pairs = (w_sizes, w2n, n2n, coords), attn.fp16_mode, norm2.eps, attn.scale, pairs
    return _Branches.apply(call, x, normed, norm2.weight, norm2.bias, *params)


def _values(layout, params, half, same):
    """What the forward made of each parameter that may have changed since, None for the others."""
    copies = iter(zip(layout.copies, layout.to))
    values = []
    for i, p in enumerate(params):
        copy, at = (None, 0) if p is None else next(copies)
        kept = None if copy is None or i in _CHECKED else same.narrow(0, copy.same, p.numel()) if copy.same >= 0 else half.narrow(0, at, p.numel())
        values.append(kept)
    return values


class _AsBefore(Function):
    """`before`, a value of the forward, with the gradient of `now`, from which it was made or is made again."""

    @staticmethod
    def forward(ctx, now, before):
        return before.to(now.dtype, copy=True).view(now.shape)

    @staticmethod
    def backward(ctx, grad):
        return grad, None


def _by_parts(call, index, x, normed, norm_weight, norm_bias, params, before, normed2_before):
    """The same through the nodes of the single layers, for gradients of gradients.  before: per parameter what the forward
    made of it, where the parameter itself may have changed since (q, k and v's scaled); normed2_before: as the forward left it."""
    channels = call.heads * call.dim
    w_sizes, w2n, n2n, coords = index
    scale = torch.ones(3 * channels, device=x.device)
    scale[:channels] = call.scale
    params = [params[0] * scale.unsqueeze(1), None if params[1] is None else params[1] * scale, *params[2:]]
    qkv_weight, qkv_bias, proj_weight, proj_bias, fc1_weight, fc1_bias, fc2_weight, fc2_bias, *tables = (
        p if b is None else _AsBefore.apply(p, b) for p, b in zip(params, before))
    qkv = _Linear.apply(normed, qkv_weight, qkv_bias)
    groups = len(tables) // 3
    kinds = [torch.cat([t.reshape(-1) for t in tables[i:i + groups]]) for i in range(0, 3 * groups, groups)]
    out = SelfAttnAIOFunction.apply(
        *qkv.view(-1, 3, call.heads, call.dim).unbind(1), *kinds, call.sizes, [None, w_sizes, None, w2n, n2n, coords], PosEmb.SEPARATE,
        TableDims.D0, IndexMode.INDIRECT, _PRECISION[call.mode])
    branch = _Linear.apply(out.reshape(-1, channels), proj_weight, proj_bias)
    norm = torch.nn.LayerNorm(channels, call.eps, elementwise_affine=False, device="meta")      # (shape and eps)
    summed, normed2 = _AddNorm.apply(x, branch, norm_weight, norm_bias, norm)
    normed2 = _AsBefore.apply(normed2, normed2_before)
    return summed, _Linear.apply(F.gelu(_Linear.apply(normed2, fc1_weight, fc1_bias)), fc2_weight, fc2_bias)


def _in_one_call(call, x, normed, norm_weight, norm_bias, given, params, layout, half, same, index):
    """(qkv, attended, its maxima and sums, sum, normed2, hidden_in, hidden_out, pending) of a block by s3d_swin_block_train, the last
    product by torch where that has bits of its own; None where one of the others' is torch's too, or where the index has to be
    looked at first."""
    (n, channels), dev = x.shape, x.device
    hidden, heads, dim, nd = call.hidden, call.heads, call.dim, len(call.sizes)
    w_sizes, w2n, n2n, coords = index
    if not (has_torchs_bits(n, 3 * channels, channels) and has_torchs_bits(n, channels, channels) and has_torchs_bits(n, hidden, channels)) \
            or w_sizes.dim() != 1 or w2n.shape != w_sizes.shape or not (n2n is None or n2n.shape == (n,)) \
            or not (x.is_contiguous() and normed.is_contiguous()) or (x.data_ptr() | normed.data_ptr()) % 16:
        return None
    last = has_torchs_bits(n, channels, hidden)
    qkv, out, normed2, hidden_in, hidden_out = (torch.empty(shape, dtype=torch.float16, device=dev) for shape in (
        (n, 3 * channels), (n, heads, dim), (n, channels), (n, hidden), (n, hidden)))
    pending = torch.empty((n, channels), dtype=torch.float16, device=dev) if last else None
    summed, omax, osum = (torch.empty(shape, dtype=torch.float32, device=dev) for shape in ((n, channels), (n, heads), (n, heads)))
    c_sizes = (ctypes.c_int32 * nd)(*call.sizes)
    p, s = _lib.BlockPass(), _lib.WindowSet()
    lib = _lib.lib()
    with _lib.on(dev):
        stream = _lib.stream(dev)
        w_sizes32, w2n32 = attn_coff._as_int32("w_sizes", w_sizes, dev), attn_coff._as_int32("w2n_indices", w2n, dev)
        n2n32 = None if n2n is None else attn_coff._as_int32("n2n_indices", n2n, dev)
        windows = w_sizes32.numel()
        plan = attn_coff._plan_for(lib, w_sizes, w2n, w_sizes32, w2n32, c_sizes, call.sizes, nd, call.table_len, n, heads, dim,
                                   _lib.S3D_DTYPE_F16, stream) if attn_coff.REUSE_PLANS else None
        s.planned = plan is not None
        if plan is None:
            plan = torch.empty(lib.s3d_attn_plan_bytes(heads, n, windows), dtype=torch.uint8, device=dev)
        s.w_sizes, s.w2n, s.n2n, s.n_coords = w_sizes32.data_ptr(), w2n32.data_ptr(), None if n2n is None else n2n32.data_ptr(), coords.data_ptr()
        s.num_windows, s.plan, s.plan_bytes = windows, plan.data_ptr(), plan.numel()
        p.params, p.copies, p.num_copies = (ctypes.c_void_p * len(given))(*[t.data_ptr() for t in given]), layout.copies, len(given)
        p.half, p.same = half.data_ptr(), None if same is None else same.data_ptr()
        places = iter(layout.to)
        (p.qkv_weight, p.qkv_bias, p.proj_weight, p.proj_bias, p.fc1_weight, p.fc1_bias, p.fc2_weight, p.fc2_bias) = (
            -1 if t is None else next(places) for t in params[:8])
        p.table_q, p.table_k, p.table_v = _table_places(layout, params)
        p.norm2_weight, p.norm2_bias, p.norm2_eps = norm_weight.data_ptr(), norm_bias.data_ptr(), call.eps
        p.x, p.normed1, p.qkv, p.attended, p.out_max, p.out_sum = (t.data_ptr() for t in (x, normed, qkv, out, omax, osum))
        p.sum, p.normed2, p.hidden_in, p.hidden_out = (t.data_ptr() for t in (summed, normed2, hidden_in, hidden_out))
        p.pending, p.windows = None if pending is None else pending.data_ptr(), ctypes.pointer(s)
        status = lib.s3d_swin_block_train(ctypes.byref(p), n, heads, dim, hidden, c_sizes, nd, call.table_len, stream)
    _lib.check(status, "s3d_swin_block_train")
    if pending is None:
        pending = F.linear(hidden_out, *_layer_copies(layout, params, half)[6:])
    return qkv, out, omax, osum, summed, normed2, hidden_in, hidden_out, pending


def _table_places(layout, params):
    """Where the query, key and value tables begin in the copies."""
    num_tables = len(params) - 8
    return layout.to[-num_tables::num_tables // 3]


def _layer_copies(layout, params, half):
    """The fp16 copies of the layers' weights and biases."""
    places, copies = iter(zip(layout.shapes, layout.to)), []
    for p in params[:8]:
        if p is None:
            copies.append(None)
            continue
        (rows, cols), at = next(places)
        copies.append(half.as_strided((rows, cols), (cols, 1), at) if p.dim() == 2 else half.as_strided((rows,), (1,), at))
    return copies


def _layer_by_layer(call, x, normed, norm_weight, norm_bias, given, params, layout, half, same, index):
    """The same by a call for each: where torch splits the sums of one of the products (few or very many rows, or many channels)."""
    n, channels = x.shape
    heads, dim, dev = call.heads, call.dim, x.device
    lib = _lib.lib()
    with _lib.on(dev):
        status = lib.s3d_half_copies((ctypes.c_void_p * len(given))(*[p.data_ptr() for p in given]), layout.copies, len(given),
                                     half.data_ptr(), None if same is None else same.data_ptr(), _lib.stream(dev))
    _lib.check(status, "s3d_half_copies")
    copies = _layer_copies(layout, params, half)
    tables = [half.as_strided((call.table_len,), (1,), at) for at in _table_places(layout, params)]
    qkv = dense_rows(normed, copies[0], copies[1])
    row = channels
    q, k, v = (qkv.as_strided((n, heads, dim), (3 * row, dim, 1), i * row) for i in range(3))
    out, omax, osum = attn_coff._attention(q, k, v, [3 * row] * 3, *tables, call.sizes, *index, True)
    branch = dense_rows(out.view(n, channels), copies[2], copies[3])
    summed, normed2 = train_add_layernorm(x, branch, norm_weight, norm_bias, call.eps)
    hidden_in = dense_rows(normed2, copies[4], copies[5])
    hidden_out = F.gelu(hidden_in)
    return qkv, out, omax, osum, summed, normed2, hidden_in, hidden_out, dense_rows(hidden_out, copies[6], copies[7])


class _Branches(Function):
    @staticmethod
    def forward(ctx, call, x, normed, norm_weight, norm_bias, *params):
        ctx.set_materialize_grads(False)
        channels, dev = x.shape[1], x.device
        given = [p for p in params if p is not None]
        # (the backward of mode 1 reads the tables in fp32)
        layout = _layout(_shapes(given), len(params) - 8, channels, call.scale, call.mode == 1)
        half = torch.empty(layout.half_count, dtype=torch.float16, device=dev)
        same = torch.empty(layout.same_count, dtype=torch.float32, device=dev) if layout.same_count else None
        (w_sizes, w2n, n2n, coords), call.index = call.index, None
        index = (w_sizes, w2n, n2n, coords)
        made = _in_one_call(call, x, normed, norm_weight, norm_bias, given, params, layout, half, same, index)
        if made is None:
            made = _layer_by_layer(call, x, normed, norm_weight, norm_bias, given, params, layout, half, same, index)
        qkv, out, omax, osum, summed, normed2, hidden_in, hidden_out, pending = made
        ctx.call, ctx.layout = call, layout
        ctx.unchecked = _unchecked(norm_bias, params)     # (leaves: their shapes, and where a replay's gradients go)
        ctx.save_for_backward(x, normed, norm_weight, qkv, out, omax, osum, summed, normed2, hidden_in, hidden_out, half, same,
                              w_sizes, w2n, n2n, coords, *(params[i] for i in _CHECKED))
        return summed, pending

    @staticmethod
    def backward(ctx, dsum, dpending):
        call, layout, needs = ctx.call, ctx.layout, ctx.needs_input_grad
        (x, normed, norm_weight, qkv, out, omax, osum, summed, normed2, hidden_in, hidden_out, half, same, w_sizes, w2n, n2n,
         coords, *checked) = ctx.saved_tensors
        norm_bias, *params = ctx.unchecked
        for i, p in zip(_CHECKED, checked):
            params.insert(i, p)
        if torch.is_grad_enabled() or dsum is None or dpending is None or not (data_only(dsum) and data_only(dpending)) \
                or dsum.dtype != torch.float32 or dpending.dtype != torch.float16:
            return _Branches._replayed(ctx, (dsum, dpending), (x, normed, norm_weight, norm_bias, *params), (w_sizes, w2n, n2n, coords),
                                       _values(layout, params, half, same), normed2)
        n, channels = x.shape
        heads, dim, dev, nd = call.heads, call.dim, x.device, len(call.sizes)
        dsum, dpending = (t if t.is_contiguous() and t.data_ptr() % 16 == 0 else t.clone(memory_format=torch.contiguous_format)
                          for t in (dsum, dpending))
        w_sizes, w2n = attn_coff._as_int32("w_sizes", w_sizes, dev), attn_coff._as_int32("w2n_indices", w2n, dev)
        n2n = None if n2n is None else attn_coff._as_int32("n2n_indices", n2n, dev)
        saved, grads = _lib.BlockSaved(), _lib.BlockGradients()
        saved.normed1, saved.qkv, saved.attended = normed.data_ptr(), qkv.data_ptr(), out.data_ptr()
        saved.out_max, saved.out_sum, saved.sum = omax.data_ptr(), osum.data_ptr(), summed.data_ptr()
        saved.normed2, saved.hidden_in, saved.hidden_out = normed2.data_ptr(), hidden_in.data_ptr(), hidden_out.data_ptr()
        base = half.data_ptr()
        saved.qkv_weight_t, saved.proj_weight_t, saved.fc1_weight_t, saved.fc2_weight_t = (base + 2 * at for at in layout.transposed if at >= 0)
        num_tables = len(params) - 8
        if same is None:
            saved.table_q, saved.table_k, saved.table_v = (base + 2 * at for at in _table_places(layout, params))
        else:
            saved.table_q, saved.table_k, saved.table_v = (same.data_ptr() + 4 * i * call.table_len for i in range(3))
        saved.norm2_weight, saved.norm2_eps = norm_weight.data_ptr(), call.eps
        saved.w_sizes, saved.w2n, saved.n2n = w_sizes.data_ptr(), w2n.data_ptr(), None if n2n is None else n2n.data_ptr()
        saved.n_coords = coords.data_ptr()
        dx, dnormed = torch.empty_like(x), torch.empty_like(normed)
        dnorm = [torch.empty_like(norm_weight), torch.empty_like(norm_bias)]
        dparams = [torch.empty_like(p) if need else None for p, need in zip(params[:8], needs[5:13])]
        dtables = [torch.empty(call.table_len, dtype=torch.float32, device=dev) for _ in range(3)]
        grads.x, grads.normed1, grads.norm2_weight, grads.norm2_bias = (t.data_ptr() for t in (dx, dnormed, *dnorm))
        (grads.qkv_weight, grads.qkv_bias, grads.proj_weight, grads.proj_bias, grads.fc1_weight, grads.fc1_bias, grads.fc2_weight,
         grads.fc2_bias) = (None if t is None else t.data_ptr() for t in dparams)
        grads.table_q, grads.table_k, grads.table_v = (t.data_ptr() for t in dtables)
        lib = _lib.lib()
        with _lib.on(dev):
            ws_bytes = lib.s3d_swin_block_grad_workspace_bytes(n, heads, dim, call.hidden, nd, call.table_len, w_sizes.numel(), call.pairs)
            workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
            status = lib.s3d_swin_block_grad(
                ctypes.byref(saved), ctypes.byref(grads), dsum.data_ptr(), dpending.data_ptr(), n, heads, dim, call.hidden,
                (ctypes.c_int32 * nd)(*call.sizes), nd, call.table_len, w_sizes.numel(), call.pairs, call.scale,
                _lib.S3D_DTYPE_F16 if same is None else _lib.S3D_DTYPE_F32_F16_ROWS, workspace.data_ptr(), ws_bytes, _lib.stream(dev))
        _lib.check(status, "s3d_swin_block_grad")
        groups = num_tables // 3
        pieces = [piece for t in dtables for piece in t.split([p.numel() for p in params[8:8 + groups]])]
        given = [dx, dnormed, *dnorm, *dparams, *(piece.view(p.shape) for piece, p in zip(pieces, params[8:]))]
        return (None, *(g if need else None for g, need in zip(given, needs[1:])))

    @staticmethod
    def _replayed(ctx, grads, inputs, index, before, normed2_before):
        """A graph of the gradients is wanted, or something follows them, or one is absent: the pass again through the
        single layers, whose backward knows these cases."""
        needs = ctx.needs_input_grad[1:]
        graph = torch.is_grad_enabled()
        with torch.enable_grad(), torch.autocast("cuda", dtype=torch.float16):
            if not graph:
                inputs = [None if t is None else t.detach().requires_grad_(need) for t, need in zip(inputs, needs)]
            outs = _by_parts(ctx.call, index, *inputs[:4], inputs[4:], before, normed2_before)
        pairs = [(o, g) for o, g in zip(outs, grads) if g is not None and o.requires_grad]
        wanted = [t for t, need in zip(inputs, needs) if need]
        if not pairs:
            return (None,) * (1 + len(needs))
        got = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs], create_graph=graph, allow_unused=True))
        return (None, *(next(got) if need else None for need in needs))

"""The tile kernels of the window attention (head_dim 16, mean window of at least 40 voxels) against the float64 oracle,
at the edges of their tiles, stages and dispatch; the other GPU files' cases run on them too where the shape says so."""
import numpy as np
import pytest
import torch

from helpers import make_attn_case, to_half_and_back

pytestmark = pytest.mark.gpu


def _case(oracle_lib, ws, cRSE, heads, dtype, fill=0.75, seed=0):
    """A dense block of 2 x 2 x 1 windows per axis pair: windows of about fill * ws^3 voxels."""
    half = (ws, ws, (ws + 1) // 2)
    n = int(fill * 8 * half[0] * half[1] * half[2])
    case = make_attn_case(oracle_lib, seed=seed + ws, n=n, ws=ws, quant=4, heads=heads, dim=16, cRSE=cRSE, extent=half)
    case.v *= np.float32(0.4)
    case.tv *= np.float32(0.2)
    if dtype == torch.float16:
        to_half_and_back(case)
    assert n >= 40 * case.index["w_sizes"].shape[0]
    return case


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("ws,cRSE,heads", [
    (8, "XYZ_RGB_NORM", 3),     # 64 rows on the position axes: a full stage
    (7, "XYZ_RGB", 2),          # an odd number of signal axes: the last stage holds one
    (5, "XYZ", 1),              # no signal axes
    (10, "XYZ", 2),             # 80 rows: beyond a stage, the sweep kernel's (also where it is the device that knows)
])
def test_forward_stages_and_row_limits(oracle_lib, hip_lib, dtype, ws, cRSE, heads):
    from gpu_helpers import assert_attn_close, run_attention
    case = _case(oracle_lib, ws, cRSE, heads, dtype)
    ref = oracle_lib.attn_fwd(*case.oracle_args(), return_stats=True)
    got, omax, osum = run_attention(case, dtype, return_stats=True)
    assert_attn_close(got, ref[0], dtype)
    assert np.allclose(omax, ref[1], rtol=0, atol=2e-5 * np.abs(ref[1]).max() if dtype == torch.float32 else 1e-3)
    assert np.allclose(osum, ref[2], rtol=1e-4 if dtype == torch.float32 else 3e-3)
    # (with statistics the sweep kernel runs, without them the tiles)
    plain = run_attention(case, dtype)
    assert_attn_close(plain, ref[0], dtype)
    assert np.array_equal(run_attention(case, dtype, device_sizes=True), plain)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("ws,fill", [(5, 0.75), (7, 0.75)])     # a tile a window, and several
def test_forward_weights_keep_their_bits(oracle_lib, hip_lib, dtype, ws, fill):
    from gpu_helpers import run_attention
    case = _case(oracle_lib, ws, "XYZ", 2, dtype, fill)
    # the rows of two axes cancel: what is left of 1000 is the rounding of the weights and of their sums in fp32.  Weights
    # of 23 bits leave 2^-24 of the 2000 that the terms' sizes add up to, and the (at most 128) terms of a sum 2^-24 each of
    # partial sums below 1000, of random sign: sqrt(128) of them at one standard deviation
    case.v[:], case.tq[:], case.tk[:] = 0, 0, 0
    for rows, value in zip(case.axis_tables(case.tv), (1000, -1000, 0)):
        rows[:] = value
    got = run_attention(case, dtype)
    assert np.abs(got).max() <= 1000 * 2.0 ** -24 * (2 + 4 * 128 ** 0.5)
    # a key of each window with a weight of e^-19 beside its value alone
    case.tv[:], case.q[:], case.k[:] = 0, 0, 0
    case.q[:, :, 0] = 1
    light = case.index["n2n"][case.index["w2n"]]
    case.k[light, :, 0], case.v[light] = -19, 30000
    got = run_attention(case, dtype)
    others = np.empty(case.N)
    others[case.index["n2n"]] = np.repeat(case.index["w_sizes"], case.index["w_sizes"]) - 1
    want = np.exp(-19.0) * 30000 / (others + np.exp(-19.0))
    want[light] = 30000 * np.exp(-19.0) / (others[light] + np.exp(-19.0))
    # fp32: 27 units of 2^-24 in the exponent (of 2) of a logit of -19, twice, and the softmax's roundings; fp16: half a unit
    # of its smallest numbers, and half of a weight's unit of 2^-39 of the sum beside 30000
    bound = 4e-6 * want if dtype == torch.float32 else 2.0 ** -25 + 30000 * 2.0 ** -40 + 1e-5 * want
    some = others > 0
    assert (np.abs(got - want[:, None, None]) <= bound[:, None, None])[some].all()


def _windows_case(oracle_lib, sizes, cRSE, heads, seed, ws=7, dim=16):
    """Windows of the given numbers of voxels, in rows of a random order."""
    from conftest import random_scene
    from helpers import AttnCase, n_coords_from_scene
    from swin3d_amd import crse, synth
    rng = np.random.default_rng(seed)
    cells = np.stack(np.meshgrid(*[np.arange(ws)] * 3, indexing="ij"), -1).reshape(-1, 3)
    coords = np.concatenate([np.concatenate([np.zeros((n, 1), np.int64), cells[rng.permutation(ws ** 3)[:n]] + [w * ws, 0, 0]], 1)
                             for w, n in enumerate(sizes)]).astype(np.int32)
    coords = coords[rng.permutation(coords.shape[0])]
    n = coords.shape[0]
    frac = rng.random((n, 3)).astype(np.float32)
    sig = rng.uniform(-1, 1, (n, crse.crse_num_axes(cRSE) - 3)).astype(np.float32)
    index, n_coords = n_coords_from_scene(oracle_lib, coords, frac, sig, 1, ws, 4, cRSE)
    assert sorted(index["w_sizes"]) == sorted(sizes)
    table_sizes = crse.crse_table_sizes(ws, 4, heads, dim, cRSE)
    q, k, v, tables = synth.layer_inputs(n, heads * dim, heads, int(sum(table_sizes)), seed=seed, recipe="sharp")
    return AttnCase(coords, 1, ws, 4, heads, dim, cRSE, index, n_coords, q, k, 0.4 * v, (0.3 * tables[0], 0.3 * tables[1], 0.2 * tables[2]),
                    table_sizes)


def _kinds(x):
    """0 finite, 1 and -1 infinite, 2 not a number"""
    return np.where(np.isnan(x), 2, np.where(np.isinf(x), np.sign(x), 0))


# units of several windows of 20, 16 and 9 voxels, windows of a tile and of several; as many voxels in larger windows that
# the mean is 40
SIZES = [20] * 5 + [16] * 4 + [9] * 8 + [64, 65, 120, 150, 150, 150, 200, 200]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("cRSE", ["XYZ", "XYZ_RGB_NORM"])
@pytest.mark.parametrize("where,value", [("q", np.nan), ("k", np.nan), ("k", np.inf), ("k masked", -np.inf), ("v", np.nan),
                                         ("v", np.inf), ("v", -np.inf), ("tq", np.inf), ("tk", np.nan), ("tv", np.inf), ("tv", np.nan)])
def test_forward_keeps_what_is_not_finite_in_its_window(oracle_lib, hip_lib, dtype, cRSE, where, value):
    """The same elements as in the oracle are NaN, plus and minus infinity and finite, and windows without such a voxel have
    the bits of a call without it."""
    from gpu_helpers import assert_attn_close, run_attention
    case = _windows_case(oracle_lib, SIZES, cRSE, 2, seed=9)
    if dtype == torch.float16:
        to_half_and_back(case)
    case.tk[:] = np.abs(case.tk)
    clean = run_attention(case, dtype)
    w_sizes, w2n, n2n = (case.index[x] for x in ("w_sizes", "w2n", "n2n"))
    touched = np.zeros(case.N, bool)
    for size in (9, 20, 64, 200):
        w = int(np.flatnonzero(w_sizes == size)[0])
        rows = n2n[w2n[w]:w2n[w] + size]
        touched[rows] = True
        if where[0] in "qkv":
            getattr(case, where[0])[rows[-1], 1, 3] = value
        if where == "k masked":
            case.q[rows, 1, 3] = np.abs(case.q[rows, 1, 3]) + 0.1
    if where[0] == "t":
        case.axis_tables(getattr(case, where))[1][5, 1, 3] = value
        touched[:] = True
    got, ref = run_attention(case, dtype), oracle_lib.attn_fwd(*case.oracle_args())
    assert np.array_equal(got[~touched], clean[~touched])
    assert np.array_equal(run_attention(case, dtype, device_sizes=True), got, equal_nan=True)
    assert not np.isfinite(got).all() or where == "k masked"
    assert np.array_equal(_kinds(got), _kinds(ref))
    same = np.isfinite(ref)
    assert_attn_close(np.where(same, got, 0), np.where(same, ref, 0), dtype)


def _backward(case, dtype, tables, dout, spare=0, part=1, forward=None):
    """forward: a list that takes the forward's results"""
    import swin3d_amd
    dev = torch.device("cuda")
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    i = case.index
    args = [t(x).to(dtype) for x in (case.q, case.k, case.v)] + [t(x) for x in (case.tq, case.tk, case.tv)]
    rest = (t(case.table_sizes), t(i["w_sizes"]), t(i["w2n"]), t(i["n2n"]), t(case.n_coords))
    out, omax, osum = swin3d_amd.window_attention_forward(*args[:3], *[x.to(dtype) for x in args[3:]], *rest, return_stats=True)
    if forward is not None:
        forward += [out, omax, osum]
    pairs = int((torch.as_tensor(i["w_sizes"]).long() ** 2).sum()) // part + spare
    return swin3d_amd.window_attention_backward(*args[:3], *[x.to(tables) for x in args[3:]], *rest, out, omax, osum,
                                                t(dout).to(dtype), pairs=pairs)


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("ws,cRSE,heads,fill", [
    (8, "XYZ_RGB_NORM", 3, 0.75),     # 64 rows on the position axes; windows of six tiles
    (7, "XYZ_RGB", 2, 0.3),           # an odd number of signal axes; windows of two tiles
    (5, "XYZ", 1, 0.2),               # no signal axes; several windows in a tile
    (10, "XYZ", 2, 0.5),              # 80 rows: beyond a stage, the pair sweeps'
])
def test_backward_stages_and_row_limits(oracle_lib, hip_lib, dtype, tables, ws, cRSE, heads, fill):
    from test_gpu_attn_bwd import _assert_close
    half = (ws, ws, (ws + 1) // 2)
    n = int(fill * 8 * half[0] * half[1] * half[2])
    case = make_attn_case(oracle_lib, seed=ws, n=n, ws=ws, quant=4, heads=heads, dim=16, cRSE=cRSE, extent=half)
    case.v *= np.float32(0.4)
    case.tv *= np.float32(0.2)
    if dtype == torch.float16:
        to_half_and_back(case)
    dout = np.random.default_rng(ws).standard_normal(case.q.shape).astype(np.float16).astype(np.float32)
    got = _backward(case, dtype, tables, dout)
    _assert_close([g.double().cpu().numpy() for g in got], oracle_lib.attn_bwd(*case.oracle_args(), dout), dtype)
    if ws == 10:
        return
    # the same bits again, also with room to spare in the store
    for again in (_backward(case, dtype, tables, dout), _backward(case, dtype, tables, dout, spare=4321)):
        assert all(torch.equal(x, y) for x, y in zip(got[:3], again[:3]))
    # too small a store: the windows beyond it and every table gradient say so
    short = _backward(case, dtype, tables, dout, part=2)
    assert all(bool(torch.isnan(g).all()) for g in short[3:])
    for g, whole in zip(short[:3], got[:3]):
        bad = torch.isnan(g.float()).flatten(1).any(1)
        assert bool(bad.any()) and torch.equal(g[~bad], whole[~bad])


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("ws,fill", [(7, 0.75), (5, 0.3)])       # several tiles a window; a tile
def test_backward_weights_keep_their_bits(oracle_lib, hip_lib, dtype, tables, ws, fill):
    """A key of each window with a weight of e^-14 / n beside every query."""
    case = _case(oracle_lib, ws, "XYZ", 2, torch.float16, fill) if fill > 0.5 else \
        to_half_and_back(make_attn_case(oracle_lib, seed=ws, n=int(fill * 1000), ws=ws, quant=4, heads=2, dim=16, cRSE="XYZ", extent=(5, 5, 3)))
    for x in (case.q, case.k, case.tq, case.tk, case.tv):
        x[:] = 0
    light = case.index["n2n"][case.index["w2n"]]
    case.q[:, :, 0], case.k[light, :, 0] = 1, -14
    dout = (1000 * (1 + np.random.default_rng(ws).random(case.q.shape))).astype(np.float16).astype(np.float32)
    ref = oracle_lib.attn_bwd(*case.oracle_args(), dout)
    dv = _backward(case, dtype, tables, dout)[2].double().cpu().numpy()[light]
    many = case.index["w_sizes"] > 1
    # fp32: 20 units of 2^-24 in the exponent (of 2), twice, and the softmax's roundings.  fp16: half of its last place, and
    # half of a weight's unit of 2^-35 beside every query's dout of at most 2000
    bound = 4e-6 * ref[2][light] + (0 if dtype == torch.float32 else
                                    2.0 ** -11 * ref[2][light] + 2000 * 2.0 ** -36 * case.index["w_sizes"][:, None, None])
    assert (np.abs(dv - ref[2][light]) <= bound)[many].all()


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
def test_backward_sums_by_row_keep_their_bits(oracle_lib, hip_lib, dtype, tables):
    """The value table's gradient under near-uniform weights: sums of either sign of weights times dout, whose error is the
    weights' own.  Of a pair: an exponential to two units of 2^-24 (in its argument, and its result) and one each of the
    logit's sum, the sum of the weights, its reciprocal and the product with it, of random sign; and the sums' own roundings,
    which the terms' sizes bound.  (Weights in units of 2^-25 left 8e-7 of the result.)"""
    case = _case(oracle_lib, 7, "XYZ_RGB_NORM", 4, torch.float16)
    for x in (case.q, case.tq, case.tk):
        x *= np.float32(2.0 ** -6)
    to_half_and_back(case)
    dout = np.random.default_rng(3).standard_normal(case.q.shape).astype(np.float16).astype(np.float32)
    got = _backward(case, dtype, tables, dout)[5].double().cpu().numpy()
    ref = np.asarray(oracle_lib.attn_bwd(*case.oracle_args(), dout)[5])
    assert np.linalg.norm(got - ref) <= 6 * 2.0 ** -24 * np.linalg.norm(ref)


def _pairwise_backward(case, out, omax, osum, dout):
    """The six gradients as sums over pairs in float64, from the forward's own results; dL is NaN where the logit is not
    finite."""
    heads, dim = case.q.shape[1:]
    q, k, v, out, dout = (torch.as_tensor(x).double().cpu() for x in (case.q, case.k, case.v, out, dout))
    omax, osum = omax.double().cpu(), osum.double().cpu()
    tables = [torch.as_tensor(t).double().view(-1, heads, dim) for t in (case.tq, case.tk, case.tv)]
    rows = [int(x) // (heads * dim) for x in case.table_sizes]
    grads = [torch.zeros_like(x) for x in (q, k, v, *tables)]
    coords = torch.as_tensor(case.n_coords)
    for w, n in zip(case.index["w2n"].tolist(), case.index["w_sizes"].tolist()):
        r, c = torch.as_tensor(case.index["n2n"][w:w + n]).long(), coords[w:w + n]
        hit = [sum(rows[:a]) + (c[:, None, a] - c[None, :, a] + float(m // 2)).clamp(0, m).long().clamp(max=m - 1) for a, m in enumerate(rows)]
        t_q, t_k, t_v = (sum(t[x] for x in hit) for t in tables)
        logit = (q[r][:, None] * (k[r][None] + t_q)).sum(-1) + (k[r][None] * t_k).sum(-1)
        p = torch.exp(logit - omax[r][:, None]) / osum[r][:, None]
        dl = (p * ((dout[r][:, None] * (v[r][None] + t_v)).sum(-1) - (dout[r] * out[r]).sum(-1)[:, None]))[..., None]
        dl[~torch.isfinite(logit)] = np.nan
        p = p[..., None]
        grads[0][r], grads[1][r] = (dl * (k[r][None] + t_q)).sum(1), (dl * (q[r][:, None] + t_k)).sum(0)
        grads[2][r] = (p * dout[r][:, None]).sum(0)
        for g, terms in zip(grads[3:], (dl * q[r][:, None], dl * k[r][None], p * dout[r][:, None])):
            for x in hit:
                g.index_put_((x.reshape(-1),), terms.reshape(-1, heads, dim), accumulate=True)
    return grads


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("where,value", [("q", np.nan), ("k", np.inf), ("v", np.nan), ("v", np.inf), ("dout", np.nan), ("dout", np.inf),
                                         ("tq", np.inf), ("tk", np.nan), ("tv", np.inf)])
def test_backward_keeps_what_is_not_finite_in_its_window(oracle_lib, hip_lib, dtype, tables, where, value):
    """What is not finite as a sum over pairs is not finite here, and nothing else but for the other channels of its voxels
    and table rows.  Windows without such a voxel have the bits of a call without it."""
    case = to_half_and_back(_windows_case(oracle_lib, SIZES, "XYZ_RGB_NORM", 2, seed=11))
    dout = np.random.default_rng(12).standard_normal(case.q.shape).astype(np.float16).astype(np.float32)
    clean = _backward(case, dtype, tables, dout)
    touched = np.zeros((case.N, 2), bool)
    for size in (9, 16, 20, 65, 200):
        w = int(np.flatnonzero(case.index["w_sizes"] == size)[0])
        rows = case.index["n2n"][case.index["w2n"][w]:case.index["w2n"][w] + size]
        touched[rows, 1] = True
        if where == "dout":
            dout[rows[4], 1, 3] = value
        elif where in "qkv":
            getattr(case, where)[rows[4], 1, 3] = value
    if where[0] == "t":
        case.axis_tables(getattr(case, where))[4][3, 1, 3] = value
        touched[:, 1] = True
    forward = []
    got = _backward(case, dtype, tables, dout, forward=forward)
    ref = _pairwise_backward(case, *forward, dout)
    scales = [max(float(r[torch.isfinite(r)].abs().max()) for r in ref[:3])] * 3 + [max(float(r[torch.isfinite(r)].abs().max()) for r in ref[3:])] * 3
    for g, before, r, scale in zip(got, clean, ref, scales):
        g = g.double().cpu().view_as(r)
        there = torch.isfinite(r).all(-1)                  # of a voxel or table row, and a head
        assert bool((~torch.isfinite(g))[~torch.isfinite(r)].all())
        if where == "tq":
            # (fp32 products make NaN of a logit of minus infinity, and of the weights of its query)
            there = there & torch.isfinite(g).all(-1)
        assert bool(torch.isfinite(g[there]).all()) and bool(there[:, 0].all())
        rel = 2e-5 if dtype == torch.float32 else 3e-3     # as elsewhere in the tests of this operator
        assert float((g - r)[there].abs().max()) <= rel * scale
        if r.shape[0] == case.N and where[0] != "t":
            assert torch.equal(g[torch.as_tensor(~touched)], before.double().cpu()[torch.as_tensor(~touched)])
    assert not all(bool(torch.isfinite(g.float()).all()) for g in got)

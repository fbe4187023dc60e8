"""The attention backward at head_dim 8 on strips (a sweep that leaves dL and P, sums over pairs by 16 voxels at a time) against
the float64 oracle: at the edges of strips and of a step of 32 keys, with what is not finite, and in its precision."""
import numpy as np
import pytest
import torch

from helpers import make_attn_case, to_half_and_back
from test_gpu_attn_tile import _backward, _pairwise_backward, _windows_case

pytestmark = pytest.mark.gpu

# strips of up to sixteen windows, of five, of two, of one; windows of a step (32), of several and beyond the pairs that a
# thread keeps (128); last strips of one voxel and full ones
SIZES = [1] * 19 + [2] * 9 + [3] * 7 + [4] * 5 + [5] * 4 + [7] * 3 + [15, 16, 16, 17, 17, 17, 20, 26, 26, 31, 32, 32, 33, 48, 63, 64, 65, 96, 129, 160, 257]
TYPES = [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)]


def _dout(case, seed):
    return np.random.default_rng(seed).standard_normal(case.q.shape).astype(np.float16).astype(np.float32)


@pytest.mark.parametrize("dtype,tables", TYPES)
@pytest.mark.parametrize("cRSE,heads", [("XYZ_RGB_NORM", 2), ("XYZ_RGB_NORM", 3), ("XYZ_RGB", 1), ("XYZ", 3)])
def test_strips_at_their_edges(oracle_lib, hip_lib, dtype, tables, cRSE, heads):
    from test_gpu_attn_bwd import _assert_close
    case = _windows_case(oracle_lib, SIZES, cRSE, heads, seed=31, dim=8)
    if dtype == torch.float16:
        to_half_and_back(case)
    dout = _dout(case, 32)
    got = _backward(case, dtype, tables, dout)
    _assert_close([g.double().cpu().numpy() for g in got], oracle_lib.attn_bwd(*case.oracle_args(), dout), dtype)
    again = _backward(case, dtype, tables, dout)
    assert all(torch.equal(x, y) for x, y in zip(got, again))       # the strips of a workgroup are fixed


@pytest.mark.parametrize("size,count", [(1, 1), (1, 16), (1, 17), (2, 41), (3, 31), (5, 20), (16, 1), (31, 3), (32, 3), (33, 3), (64, 2), (65, 2), (300, 1)])
def test_a_single_window_size(oracle_lib, hip_lib, size, count):
    from test_gpu_attn_bwd import _assert_close
    case = _windows_case(oracle_lib, [size] * count, "XYZ", 1, seed=size, dim=8)
    dout = _dout(case, size)
    got = _backward(case, torch.float32, torch.float32, dout)
    _assert_close([g.double().cpu().numpy() for g in got], oracle_lib.attn_bwd(*case.oracle_args(), dout), torch.float32)


@pytest.mark.parametrize("dtype,tables", TYPES)
@pytest.mark.parametrize("where,value", [("q", np.nan), ("k", np.inf), ("v", np.nan), ("dout", np.nan), ("dout", np.inf), ("tq", np.inf), ("tk", np.nan), ("tv", np.inf)])
def test_what_is_not_finite_stays_in_its_window(oracle_lib, hip_lib, dtype, tables, where, value):
    """As at head_dim 16: what is not finite as a sum over pairs is not finite here, windows without such a voxel keep their
    bits."""
    case = to_half_and_back(_windows_case(oracle_lib, SIZES, "XYZ_RGB_NORM", 2, seed=33, dim=8))
    dout = _dout(case, 34)
    clean = _backward(case, dtype, tables, dout)
    touched = np.zeros((case.N, 2), bool)
    for size in (7, 16, 26, 65):
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
        there = torch.isfinite(r).all(-1)
        assert bool((~torch.isfinite(g))[~torch.isfinite(r)].all())
        if where == "tq":
            there = there & torch.isfinite(g).all(-1)      # (products with an infinity make NaN of a logit of minus infinity)
        assert bool(torch.isfinite(g[there]).all()) and bool(there[:, 0].all())
        rel = 2e-5 if dtype == torch.float32 else 3e-3     # as elsewhere in the tests of this operator
        assert float((g - r)[there].abs().max()) <= rel * scale
        if r.shape[0] == case.N and where[0] != "t":
            assert torch.equal(g[torch.as_tensor(~touched)], before.double().cpu()[torch.as_tensor(~touched)])


@pytest.mark.parametrize("dtype,tables", TYPES)
def test_sums_by_row_keep_their_bits(oracle_lib, hip_lib, dtype, tables):
    """The value table's gradient under near-uniform weights: of a pair, the roundings of its weight (an exponential to two
    units of 2^-24, one each of the logit's sum, the sum of the weights, its reciprocal and the product), of random sign."""
    case = make_attn_case(oracle_lib, seed=35, n=3000, ws=5, quant=4, heads=4, dim=8, cRSE="XYZ_RGB_NORM", extent=(16, 16, 8))
    for x in (case.q, case.tq, case.tk):
        x *= np.float32(2.0 ** -6)
    to_half_and_back(case)
    dout = _dout(case, 36)
    got = _backward(case, dtype, tables, dout)[5].double().cpu().numpy()
    ref = np.asarray(oracle_lib.attn_bwd(*case.oracle_args(), dout)[5])
    assert np.linalg.norm(got - ref) <= 6 * 2.0 ** -24 * np.linalg.norm(ref)


@pytest.mark.parametrize("dtype,tables", TYPES)
@pytest.mark.parametrize("dim", [8, 16])
def test_keys_of_little_weight_keep_their_bits(oracle_lib, hip_lib, dtype, tables, dim):
    """dv of keys whose weights are e^-7 to e^-22 in every query, under a gradient as large as a loss scale makes it.  A weight's
    relative error is that of its logit, up to 22 in some twenty roundings of 2^-24, and of an exponential: 2^-14 of the terms'
    sizes; the result is rounded to its type."""
    case = _windows_case(oracle_lib, SIZES, "XYZ_RGB", 2, seed=37, dim=dim)
    rng = np.random.default_rng(38)
    for x in (case.q, case.k, case.tq, case.tk):
        x *= np.float32(2.0 ** -3)
    light = rng.random(case.N) < 0.4
    case.q[:, :, 0] = 1
    case.k[light, :, 0] = -rng.uniform(7, 22, (int(light.sum()), 1))
    to_half_and_back(case)
    dout = (8192 * rng.standard_normal(case.q.shape)).astype(np.float16).astype(np.float32)
    forward = []
    got = _backward(case, dtype, tables, dout, forward=forward)[2].double().cpu()
    ref, size = (_pairwise_backward(case, *forward, x)[2] for x in (dout, np.abs(dout)))
    bound = 2.0 ** -14 * size + (2.0 ** -11 * ref.abs() + 2.0 ** -25 if dtype == torch.float16 else 0)
    assert bool(((got.view_as(ref) - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype,tables", TYPES)
@pytest.mark.parametrize("cRSE,value", [("XYZ_RGB_NORM", np.inf), ("XYZ_RGB", np.nan), ("XYZ", -np.inf)])
def test_a_channel_of_dout_that_is_not_finite_stays_one(oracle_lib, hip_lib, dtype, tables, cRSE, value):
    """A dout with a channel that is not finite spoils that channel of dv in its window, and of dTv in the rows of its pairs: the
    others are the sums over pairs that they are without it."""
    case = to_half_and_back(_windows_case(oracle_lib, SIZES, cRSE, 3, seed=39, dim=8))
    dout = _dout(case, 40)
    clean = _backward(case, dtype, tables, dout)
    touched = np.zeros((case.N, 3), bool)
    for i, size in enumerate((1, 3, 7, 26, 32, 65, 160, 257)):
        w = int(np.flatnonzero(case.index["w_sizes"] == size)[0])
        rows = case.index["n2n"][case.index["w2n"][w]:case.index["w2n"][w] + size]
        touched[rows, i % 3] = True
        dout[rows[size // 2], i % 3, i % 2 + 3] = value
    forward = []
    got = _backward(case, dtype, tables, dout, forward=forward)
    ref = _pairwise_backward(case, *forward, dout)
    dv, want = got[2].double().cpu(), ref[2]
    assert torch.equal(dv.isnan(), want.isnan()) and torch.equal(dv.isinf(), want.isinf())
    there = torch.isfinite(want)
    rel = 2e-5 if dtype == torch.float32 else 3e-3         # as elsewhere in the tests of this operator
    assert float((dv - want)[there].abs().max()) <= rel * float(want[there].abs().max())
    rest = torch.as_tensor(~touched)
    assert torch.equal(dv[rest], clean[2].double().cpu()[rest])
    dtv, want = got[5].double().cpu().view_as(ref[5]), ref[5]
    assert torch.equal(~torch.isfinite(dtv), ~torch.isfinite(want)) and not torch.isfinite(dtv[..., 3:5]).all() \
        and bool(torch.isfinite(dtv[..., [0, 1, 2, 5, 6, 7]]).all())
    there = torch.isfinite(want)
    assert float((dtv - want)[there].abs().max()) <= rel * float(want[there].abs().max())
    again = _backward(case, dtype, tables, dout)
    assert all(torch.equal(x.nan_to_num(1.0, 2.0, 3.0), y.nan_to_num(1.0, 2.0, 3.0)) for x, y in zip(got, again))

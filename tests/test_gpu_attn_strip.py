"""The strip kernels of the attention backward (sums over pairs, 16 voxels of windows of one size at a time) against the
float64 oracle, at the edges of their strips: windows that share one, that fill one, of every number of steps."""
import numpy as np
import pytest
import torch

from helpers import to_half_and_back
from test_gpu_attn_tile import _backward, _windows_case

pytestmark = pytest.mark.gpu

# strips of up to sixteen windows, of two, of one; windows of one to five steps of 32 voxels and beyond the pairs that a
# thread keeps (128); a last strip of one voxel (33 = 2 * 16 + 1, 65, 129, 257) and a full one
SIZES = [1] * 19 + [2] * 9 + [3] * 7 + [5] * 4 + [15, 16, 16, 17, 17, 17, 31, 32, 33, 48, 49, 49, 49, 63, 64, 65, 96, 97, 128, 129, 160, 257]


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("cRSE,heads", [("XYZ_RGB_NORM", 2), ("XYZ_RGB", 1), ("XYZ", 3)])
def test_strips_at_their_edges(oracle_lib, hip_lib, dtype, tables, cRSE, heads):
    from test_gpu_attn_bwd import _assert_close
    case = _windows_case(oracle_lib, SIZES, cRSE, heads, seed=21)
    if dtype == torch.float16:
        to_half_and_back(case)
    dout = np.random.default_rng(22).standard_normal(case.q.shape).astype(np.float16).astype(np.float32)
    got = _backward(case, dtype, tables, dout)
    _assert_close([g.double().cpu().numpy() for g in got], oracle_lib.attn_bwd(*case.oracle_args(), dout), dtype)
    again = _backward(case, dtype, tables, dout)
    assert all(torch.equal(x, y) for x, y in zip(got, again))       # table gradients too: the strips of a workgroup are fixed


@pytest.mark.parametrize("size,count", [(1, 1), (1, 16), (1, 17), (16, 1), (7, 60), (300, 1)])
def test_a_single_window_size(oracle_lib, hip_lib, size, count):
    from test_gpu_attn_bwd import _assert_close
    case = _windows_case(oracle_lib, [size] * count, "XYZ", 1, seed=size)
    dout = np.random.default_rng(size).standard_normal(case.q.shape).astype(np.float32)
    got = _backward(case, torch.float32, torch.float32, dout)
    _assert_close([g.double().cpu().numpy() for g in got], oracle_lib.attn_bwd(*case.oracle_args(), dout), torch.float32)

"""dL and P of every pair on strips (fp16 features, head_dim 16) through the six gradients, against the float64 oracle, at the
edges of strips of 16 queries, steps of 32 keys and blocks of 96."""
import numpy as np
import pytest
import torch

from helpers import to_half_and_back
from test_gpu_attn_tile import _backward, _windows_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tables", [torch.float16, torch.float32])
@pytest.mark.parametrize("cRSE,heads,sizes", [
    ("XYZ_RGB_NORM", 2, [1, 15, 16, 17, 32, 33, 64, 65, 95, 96, 97, 192, 193, 343]), ("XYZ_RGB", 3, [31, 48, 97, 200]),
    ("XYZ", 1, [2, 96, 129]), ("XYZ", 1, [1]), ("XYZ", 40, [20] * 40),      # (the last: more strips than places)
])
def test_gradients_at_the_edges(oracle_lib, hip_lib, tables, cRSE, heads, sizes):
    from test_gpu_attn_bwd import _assert_close
    case = to_half_and_back(_windows_case(oracle_lib, sizes, cRSE, heads, seed=3))
    dout = np.random.default_rng(5).standard_normal(case.q.shape).astype(np.float16).astype(np.float32)
    got = _backward(case, torch.float16, tables, dout)
    _assert_close([g.double().cpu().numpy() for g in got], oracle_lib.attn_bwd(*case.oracle_args(), dout), torch.float16)
    assert all(torch.equal(x, y) for x, y in zip(got[:3], _backward(case, torch.float16, tables, dout, spare=777)[:3]))

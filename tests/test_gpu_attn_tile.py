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
    assert np.array_equal(run_attention(case, dtype, device_sizes=True), got)

"""The forward's work list handed out to wavefronts: launches of fewer units than workgroups, than wavefronts, of one to two a
wavefront (whose first units are the wavefronts' own) and of more (all by tickets), against the CPU oracle, and the bits of a call
that follows on the same list."""
import numpy as np
import pytest
import torch

from helpers import make_attn_case, to_half_and_back

pytestmark = pytest.mark.gpu


# voxels, heads, head_dim, extent: with 256 CUs and twelve wavefronts each, 3072 wavefronts share the head groups
@pytest.mark.parametrize("n,heads,dim,extent", [
    (1, 1, 8, (4, 4, 4)),                # one unit, 255 workgroups without any
    (70, 3, 8, (8, 8, 4)),
    (900, 5, 16, (14, 14, 14)),          # five head groups: an odd number of workgroups each
    (6000, 6, 8, (30, 30, 24)),
    (9000, 40, 16, (33, 33, 28)),        # 20 head groups of twelve workgroups
    (60000, 6, 8, (72, 72, 40)),         # about as many units as wavefronts
    (130000, 6, 8, (92, 92, 52)),        # and twice as many
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_every_unit_is_done_once(oracle_lib, hip_lib, n, heads, dim, extent, dtype):
    from gpu_helpers import run_attention, assert_attn_close
    if dtype == torch.float32 and n > 60000:
        pytest.skip("the same list as in fp16")
    case = make_attn_case(oracle_lib, seed=61, n=n, ws=5, quant=4, heads=heads, dim=dim, cRSE="XYZ_RGB", extent=extent, recipe="layer")
    if dtype == torch.float16:
        to_half_and_back(case)
    got = run_attention(case, dtype)
    assert_attn_close(got, oracle_lib.attn_fwd(*case.oracle_args()), dtype)
    assert np.array_equal(run_attention(case, dtype), got)

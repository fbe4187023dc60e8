"""The strip kernel of the window attention forward (fp16, head_dim 16, launches of few strips) against the float64 oracle, at
the edges of its strips of 16 queries and blocks of 64 keys, and on either side of its dispatch."""
import numpy as np
import pytest
import torch

from helpers import to_half_and_back
from test_gpu_attn_tile import _windows_case

pytestmark = pytest.mark.gpu

# a strip, two, a full block of keys, two blocks, three and six of them
EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 96, 127, 128, 129, 200, 343]
SMALL = [3, 5, 8, 13, 1, 21]


@pytest.mark.parametrize("cRSE,heads,sizes", [
    ("XYZ_RGB_NORM", 3, EDGES), ("XYZ_RGB", 2, EDGES), ("XYZ", 1, EDGES),
    ("XYZ_RGB_NORM", 24, [98]), ("XYZ_RGB_NORM", 1, [1]),
    ("XYZ", 2, SMALL * 10),                    # a mean window below the rule's
    ("XYZ", 40, [64] * 25),                    # 5000 strips at most: more than one a workgroup
    ("XYZ", 40, [64] * 40),                    # beyond the rule: the sweep's
    ("XYZ_RGB", 40, [64] * 32), ("XYZ_RGB_NORM", 40, [64] * 32), ("XYZ_RGB_NORM", 40, [64] * 37),      # 6400: with nine axes strips; 7400
    ("XYZ", 1, [5, 9] * 128), ("XYZ", 1, [5, 9] * 128 + [7]),      # windows whose lists one launch makes, and one more
])
def test_strips_of_every_size(oracle_lib, hip_lib, cRSE, heads, sizes):
    from gpu_helpers import assert_attn_close, run_attention
    case = to_half_and_back(_windows_case(oracle_lib, sizes, cRSE, heads, seed=len(sizes)))
    got, ref = run_attention(case, torch.float16), oracle_lib.attn_fwd(*case.oracle_args())
    assert_attn_close(got, ref, torch.float16)
    assert_attn_close(run_attention(case, torch.float16, return_stats=True)[0], ref, torch.float16)      # (the sweep's, on a plan like it)
    assert np.array_equal(run_attention(case, torch.float16), got)
    assert np.array_equal(run_attention(case, torch.float16, device_sizes=True), got)


def test_error_is_no_larger_than_the_sweeps(oracle_lib, hip_lib):
    """What is left of a result in fp16 is its own rounding, half of 2^-10 to 2^-11 of it uniformly: 2^-11 / sqrt(3) = 2.8e-4
    at the most; sums in fp16, as the sweep's of three value rows, would add as much."""
    from gpu_helpers import run_attention
    case = to_half_and_back(_windows_case(oracle_lib, [49] * 6 + [91] * 3, "XYZ_RGB_NORM", 2, seed=4))
    ref = np.asarray(oracle_lib.attn_fwd(*case.oracle_args()))
    strips, sweep = (run_attention(case, torch.float16), run_attention(case, torch.float16, return_stats=True)[0])
    error = [np.linalg.norm(x - ref) / np.linalg.norm(ref) for x in (strips, sweep)]
    assert error[0] <= 2.0 ** -11 / 3 ** 0.5 and error[0] <= error[1]


@pytest.mark.parametrize("dtype,windows", [(torch.float16, 32), (torch.float32, 120)])
@pytest.mark.parametrize("order", [(6, 9, 3), (9, 6, 9)])
def test_plans_of_calls_with_more_or_fewer_axes(hip_lib, dtype, windows, order):
    """One window set, table sizes on the device, between the lines for six axes and for nine: a plan has the lists of its own call."""
    from swin3d_amd import window_attention_forward
    gen = torch.Generator("cuda").manual_seed(windows)
    heads, n = 40, 64 * windows
    w_sizes = torch.full((windows,), 64, dtype=torch.int32, device="cuda")
    w2n = (w_sizes.cumsum(0) - w_sizes).int()
    n2n = torch.randperm(n, device="cuda", generator=gen).int()
    q, k, v = (torch.randn(n, heads, 16, device="cuda", generator=gen).to(dtype) for _ in range(3))
    for axes in order:
        sizes = [20 * heads * 16] * axes
        tables = [(0.1 * torch.randn(sum(sizes), device="cuda", generator=gen)).to(dtype) for _ in range(3)]
        coords = 10 * torch.rand(n, axes, device="cuda", generator=gen)
        got = window_attention_forward(0.25 * q, k, v, *tables, torch.tensor(sizes, dtype=torch.int32, device="cuda"), w_sizes, w2n, n2n, coords)
        want = window_attention_forward(0.25 * q, k, v, *tables, sizes, w_sizes.clone(), w2n, n2n, coords)
        assert torch.equal(got, want) and bool(got.isfinite().all()), axes

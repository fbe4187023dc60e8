"""The forward's work list handed out to wavefronts: launches of fewer units than wavefronts, whose units are the wavefronts' own, of one to
two a wavefront, whose first units are and the others go by tickets, and of more, all by tickets.  One plan, three launches, each into an
output of NaN, against the CPU oracle: every unit is done, and a launch leaves the counters at zero for the next."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import make_attn_case, to_half_and_back

pytestmark = pytest.mark.gpu

QUEUES, COUNTER_STRIDE = 8, 64        # of the plan: a head's counters, that many ints apart, then the number of units


def _heads_a_wavefront(dtype, heads, dim):
    if dtype == torch.float16 and dim <= 16:
        return 3 if dim == 8 and heads % 3 == 0 else 2 if heads % 2 == 0 else 1
    return 2 if dim == 8 and heads % 2 == 0 else 1


def _wavefronts(dtype, heads, dim):
    """wavefronts that serve a head group: workgroups a CU by their wavefronts, shared by the groups"""
    on_cu, waves = (1, 12) if dim <= 16 else (2, 4) if dtype == torch.float16 else (1, 8)
    groups = heads // _heads_a_wavefront(dtype, heads, dim)
    return on_cu * torch.cuda.get_device_properties(0).multi_processor_count // groups * waves


FEW, OWN, TICKETS = (0, 1), (1, 2), (2, 10)


# voxels, heads, head_dim, extent, units a wavefront in fp16 and in fp32 with 256 CUs
@pytest.mark.parametrize("n,heads,dim,extent,half,full", [
    (1, 1, 8, (4, 4, 4), FEW, FEW),                 # one unit, 255 workgroups without any
    (70, 3, 8, (8, 8, 4), FEW, FEW),
    (900, 5, 16, (14, 14, 14), FEW, FEW),           # five head groups: an odd number of workgroups each
    (6000, 6, 8, (30, 30, 24), FEW, FEW),
    (24000, 6, 8, (50, 50, 34), FEW, OWN),          # 0.98 and 1.47; fp32: 85 workgroups a group, so queues of 11 and of 10
    (30000, 6, 8, (56, 56, 36), OWN, OWN),          # 1.22 and 1.84
    (20000, 5, 16, (46, 46, 34), OWN, OWN),         # 1.96; 51 workgroups a group
    (12000, 12, 16, (38, 38, 30), OWN, TICKETS),
    (12000, 4, 32, (38, 38, 30), OWN, OWN),         # two workgroups of four wavefronts a CU, and one of eight
    (9000, 40, 16, (33, 33, 28), TICKETS, TICKETS),     # 20 head groups of twelve workgroups, 40 of six
    (60000, 6, 8, (72, 72, 40), TICKETS, TICKETS),      # 2.2 and 3.2
    (130000, 6, 8, (92, 92, 52), TICKETS, TICKETS),     # 3.3 and 4.6
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_every_unit_is_done_once(oracle_lib, hip_lib, n, heads, dim, extent, half, full, dtype):
    from gpu_helpers import assert_attn_close
    from swin3d_amd import _lib
    case = make_attn_case(oracle_lib, seed=61, n=n, ws=5, quant=4, heads=heads, dim=dim, cRSE="XYZ_RGB", extent=extent, recipe="layer")
    if dtype == torch.float16:
        to_half_and_back(case)
    ref, rmax, _, _ = oracle_lib.attn_fwd(*case.oracle_args(), return_stats=True)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    q, k, v, tq, tk, tv = (t(x).to(dtype) for x in (case.q, case.k, case.v, case.tq, case.tk, case.tv))
    w_sizes, w2n, n2n = (t(case.index[x]).int() for x in ("w_sizes", "w2n", "n2n"))
    n_coords = t(case.n_coords)
    sizes = (ctypes.c_int32 * len(case.table_sizes))(*[int(x) for x in case.table_sizes])
    shape = (n, heads, dim, w_sizes.numel())
    code = _lib.S3D_DTYPE_F16 if dtype == torch.float16 else _lib.S3D_DTYPE_F32
    stream = torch.cuda.current_stream().cuda_stream
    plan = torch.empty(hip_lib.s3d_attn_plan_bytes(heads, n, w_sizes.numel()), dtype=torch.uint8, device="cuda")
    _lib.check(hip_lib.s3d_attn_plan(sizes, len(sizes), tq.numel(), w_sizes.data_ptr(), w2n.data_ptr(), *shape, code, plan.data_ptr(),
                                     plan.numel(), stream), "s3d_attn_plan")
    counters = plan[:4 * heads * QUEUES * COUNTER_STRIDE].view(torch.int32)[::COUNTER_STRIDE]
    units = int(plan[4 * heads * QUEUES * COUNTER_STRIDE:][:4].view(torch.int32))
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        low, high = half if dtype == torch.float16 else full
        assert low < units / _wavefronts(dtype, heads, dim) <= high
    first = None
    for _ in range(3):
        # (a call that asks for the softmax's statistics is the sweep's, whatever its size)
        out, omax, osum = (torch.full(s, float("nan"), dtype=d, device="cuda")
                           for s, d in ((q.shape, dtype), (q.shape[:2], torch.float32), (q.shape[:2], torch.float32)))
        _lib.check(hip_lib.s3d_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), tq.data_ptr(), tk.data_ptr(), tv.data_ptr(), sizes,
                                        len(sizes), tq.numel(), w_sizes.data_ptr(), w2n.data_ptr(), n2n.data_ptr(), n_coords.data_ptr(),
                                        out.data_ptr(), omax.data_ptr(), osum.data_ptr(), *shape, 0, code, _lib.S3D_ATTN_PLANNED,
                                        plan.data_ptr(), plan.numel(), stream), "s3d_attn_fwd")
        torch.cuda.synchronize()
        assert not counters.any()
        if first is None:
            first = out, omax, osum
            assert_attn_close(out.double().cpu().numpy(), ref, dtype)
            assert np.abs(omax.double().cpu().numpy() - rmax).max() <= 1e-4 * max(1.0, np.abs(rmax).max())
        assert all(torch.equal(x, y) for x, y in zip((out, omax, osum), first))

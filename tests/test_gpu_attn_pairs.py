"""The backward's pair sweeps, whose key-owned half reads the other's records in runs, against the fused sweeps that keep none:
windows on both sides of the runs of four records and of the lanes that share a key, in stores with nothing behind them."""
import numpy as np
import pytest
import torch

from swin3d_amd.sparse_dl.attn.attn_coff import window_attention_backward, window_attention_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [3], [2, 1, 3], [4, 5, 7, 8, 9, 1], [31, 32, 33, 34], [63, 64, 65, 66, 2], [127, 128, 129, 130],
                                   [257, 515, 3], [5] * 700 + [26] * 300 + [1]])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("heads,dim,rows", [(3, 8, 40), (2, 16, 60)])       # (60 rows on a signal axis: not on tiles)
def test_pair_sweeps_against_the_fused(hip_lib, sizes, dtype, heads, dim, rows):
    gen = torch.Generator(device="cuda").manual_seed(len(sizes) + sizes[0])
    rand = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)
    w_sizes = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    w2n = (w_sizes.cumsum(0) - w_sizes).int()
    n = sum(sizes)
    n2n = torch.randperm(n, device="cuda", generator=gen).int()
    coords = torch.rand(n, 6, device="cuda", generator=gen) * (rows // 2)
    table_sizes = [rows * heads * dim] * 6
    q, k, v, dout = (rand(n, heads, dim).to(dtype) for _ in range(4))
    q = q * dim ** -0.5
    tables = [(rand(sum(table_sizes)) * 0.2).to(dtype) for _ in range(3)]
    index = (table_sizes, w_sizes, w2n, n2n, coords)
    out, top, total = window_attention_forward(q, k, v, *tables, *index, return_stats=True)
    args = (q, k, v, *tables, *index, out, top, total, dout)
    for at, (got, want) in enumerate(zip(window_attention_backward(*args), window_attention_backward(*args, pairs=0))):
        # rounded results of the same fp32 products: one place of the features' type, or fp32 sums in another order; the fused
        # sweeps add the table rows of fp16 in another grouping (two roundings of 2^-11 more on a third of the sum)
        bound = 1e-5 if dtype == torch.float32 else 2e-3
        assert got.dtype == want.dtype and bool(got.isfinite().all())
        assert float((got.float() - want.float()).abs().max()) <= bound * float(want.float().abs().max() + 1e-6), at


def _call(sizes, dtype, tables_dtype, heads, dim, rows, seed):
    """(arguments of the backward) for windows of `sizes` voxels and tables of `rows` rows an axis."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)
    w_sizes = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    w2n = (w_sizes.cumsum(0) - w_sizes).int()
    n = sum(sizes)
    n2n = torch.randperm(n, device="cuda", generator=gen).int()
    coords = torch.rand(n, len(rows), device="cuda", generator=gen) * (torch.tensor(rows, device="cuda") // 2)
    table_sizes = [r * heads * dim for r in rows]
    q, k, v, dout = (rand(n, heads, dim).to(dtype) for _ in range(4))
    q = q * dim ** -0.5
    tables = [rand(sum(table_sizes)) * 0.2 for _ in range(3)]
    index = (table_sizes, w_sizes, w2n, n2n, coords)
    out, top, total = window_attention_forward(q, k, v, *[t.to(dtype) for t in tables], *index, return_stats=True)
    return (q, k, v, *[t.to(tables_dtype) for t in tables], *index, out, top, total, dout)


def _assert_same_sums(got, want, dtype):
    """Of dq, dk, dv and of the table gradients, to the largest of the three (see test_gpu_attn_bwd.py)."""
    bound = 2e-5 if dtype == torch.float32 else 3e-3
    for group in (slice(0, 3), slice(3, 6)):
        largest = max(float(w.float().abs().max()) for w in want[group])
        for at, (g, w) in enumerate(zip(got[group], want[group])):
            assert g.dtype == w.dtype and bool(g.isfinite().all()) and float((g.float() - w.float()).abs().max()) <= bound * largest, at


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("heads,rows", [(2, [70] * 3 + [20] * 6), (6, [66] * 3 + [30] * 6), (5, [40] * 9), (40, [40] * 6), (4, [40] * 6), (3, [70, 60, 60])])
def test_narrow_heads_with_tables_that_no_strip_takes(hip_lib, dtype, tables, heads, rows):
    """head_dim 8, up to 64 rows an axis on average (beyond, the general form adds in any order): heads in pairs and by themselves,
    three to nine axes, head groups in whole sets and in turn, fp32 tables beside fp16 features; windows where the sweeps change
    their lanes and begin to cut them into chunks of 64."""
    sizes = [1, 16, 31, 32, 33, 63, 64, 65, 127, 128, 129, 192, 193] + [5] * 40 + [26] * 20
    args = _call(sizes, dtype, tables, heads, 8, rows, heads)
    got = window_attention_backward(*args)
    _assert_same_sums(got, window_attention_backward(*args, pairs=0), dtype)
    assert all(torch.equal(a, b) for a, b in zip(got[:3], window_attention_backward(*args)[:3]))


@pytest.mark.parametrize("voxels", [41_600, 41_700])
@pytest.mark.parametrize("axes", [9, 6])
def test_first_level_in_fp32(hip_lib, voxels, axes):
    """6 heads of 8 on either side of 250,000 (voxel, head): up to there fp32 runs on strips, beyond on the sweeps, whose queues then
    have more units than wavefronts."""
    sizes = np.random.default_rng(axes).integers(1, 52, voxels // 26).tolist()
    sizes += [26] * ((voxels - sum(sizes)) // 26) if sum(sizes) < voxels else []
    while sum(sizes) > voxels:
        sizes.pop()
    sizes += [1] * (voxels - sum(sizes))
    args = _call(sizes, torch.float32, torch.float32, 6, 8, [40] * 3 + [16] * (axes - 3), voxels)
    got = window_attention_backward(*args)
    _assert_same_sums(got, window_attention_backward(*args, pairs=0), torch.float32)
    again = window_attention_backward(*args)
    assert all(torch.equal(a, b) for a, b in zip(got[:3], again[:3]))
    assert all(float((a - b).abs().max()) <= 1e-5 * float(a.abs().max()) for a, b in zip(got[3:], again[3:]))

"""The backward's pair sweeps, whose key-owned half reads the other's records in runs, against the fused sweeps that keep none:
windows on both sides of the runs of four records and of the lanes that share a key, in stores with nothing behind them."""
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

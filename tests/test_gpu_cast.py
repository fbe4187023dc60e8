"""Casts of several arrays in one launch, bit for bit the framework's; the attention backward on rows apart."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1], [3, 4, 5], [1023, 1024, 1025, 100_003], [7] * 17, [2_000_000, 1]])
def test_cast_half(hip_lib, counts):
    from swin3d_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(1)
    some = [torch.randn(c, device="cuda", generator=gen) * 10 ** (i % 5 - 2) for i, c in enumerate(counts)]
    some[0][0] = 7e4
    if counts[0] > 2:
        some[0][1:3] = torch.tensor([float("nan"), 3e-8], device="cuda")
    some.append(torch.randn(40, device="cuda", generator=gen)[1:])         # not aligned
    for got, t in zip(_lib.cast_half(some), some):
        assert torch.equal(got.view(torch.int16), t.half().view(torch.int16))


@pytest.mark.parametrize("dtype,tables", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("dim,window", [(8, 5), (16, 7), (16, 5), (32, 5)])       # pair sweeps, strips; head_dim 32: the general form
def test_backward_reads_rows_apart(oracle_lib, hip_lib, dtype, tables, dim, window):
    """Slices of a projection's output give the gradients of dense copies, to the bit for dq, dk, dv."""
    from helpers import make_attn_case
    from swin3d_amd.sparse_dl.attn.attn_coff import _attention_backward, window_attention_forward
    if dim == 32 and dtype != tables:
        pytest.skip("the general form's types are tested elsewhere")
    case = make_attn_case(oracle_lib, seed=dim, n=900, ws=window, quant=4, heads=3, dim=dim, cRSE="XYZ_RGB", extent=(2 * window,) * 2 + (window,))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    i = case.index
    qkv = torch.stack([t(x) for x in (case.q, case.k, case.v)], 1).to(dtype)
    parts = [qkv[:, s] for s in range(3)]
    rest = (t(case.table_sizes), t(i["w_sizes"]), t(i["w2n"]), t(i["n2n"]), t(case.n_coords))
    flat = [t(x) for x in (case.tq, case.tk, case.tv)]
    out, omax, osum = window_attention_forward(*parts, *[x.to(dtype) for x in flat], *rest, return_stats=True)
    dout = torch.randn(out.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)).to(dtype)
    args = [x.to(tables) for x in flat], rest, (out, omax, osum, dout, None)
    apart = _attention_backward(*parts, *args[0], *args[1], *args[2], True)
    dense = _attention_backward(*[x.contiguous() for x in parts], *args[0], *args[1], *args[2], False)
    for at, (x, y) in enumerate(zip(apart, dense)):
        if at < 3 and dim < 32:
            assert torch.equal(x, y)
        else:
            # fp32 sums whose order differs between calls (head_dim 32: dk and dv by atomics, rounded to the features' type)
            bound = 2 ** -10 if at < 3 and dtype == torch.float16 else 1e-5
            assert float((x.float() - y.float()).abs().max()) <= bound * float(y.float().abs().max())
    with pytest.raises(RuntimeError, match="contiguous"):
        _attention_backward(*parts, *args[0], *args[1], *args[2], False)

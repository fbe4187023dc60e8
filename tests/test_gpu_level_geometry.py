"""A level's geometry in one kernel a step against the tensor statements, to the bit."""
import numpy as np
import pytest
import torch

from conftest import random_scene

pytestmark = pytest.mark.gpu


def _level(seed, n, stride, columns, extent=(24, 24, 12), batches=2):
    rng = np.random.default_rng(seed)
    coords = torch.from_numpy(random_scene(rng, n, extent=extent, batches=batches, stride=stride)).cuda()
    coords = coords[torch.argsort(coords[:, 0], stable=True)].contiguous()
    n = coords.shape[0]
    signals = torch.from_numpy(rng.uniform(-1, 1, (n, columns)).astype(np.float32)).cuda()
    signals[:, 0] = coords[:, 0].float()
    signals[:, 1:4] = coords[:, 1:].float() + stride * torch.rand((n, 3), device="cuda")
    return coords, signals


@pytest.mark.parametrize("n,stride,columns,factor", [(1, 1, 4, 2), (5000, 2, 10, 2), (3000, 1, 7, 3), (4000, 3, 16, 4), (2000, 1, 10, 5)])
def test_pooled_level(hip_lib, n, stride, columns, factor):
    from swin3d_amd import encoder
    from swin3d_amd.window_index import build_window_indices
    coords, signals = _level(n, n, stride, columns)
    signals[:: 7] = signals[0].clone()                             # ties
    index = build_window_indices(coords, stride, factor, (0,))[0]
    wide = torch.cat([signals, signals], 1)[:, :columns]   # rows apart
    coarse, coarse_signals = encoder._pool_level(coords, stride * factor, wide, index)
    want, pick = encoder.pool_and_pick(coords, stride, factor, signals, index)
    assert torch.equal(coarse, want) and torch.equal(coarse_signals, signals[pick])


@pytest.mark.parametrize("n,stride,window,others", [(1, 1, 5, 0), (5000, 2, 5, 6), (3000, 3, 7, 3)])
def test_level_signals(hip_lib, n, stride, window, others):
    from swin3d_amd import encoder
    from swin3d_amd.window_index import build_window_indices, window_signals
    coords, signals = _level(n + window, n, stride, 10)
    for index in build_window_indices(coords, stride, window, (0, window // 2)):
        got = encoder._level_signals(index, coords, stride, signals, others, 4)
        want = window_signals(index, *encoder._local_and_extra(coords, stride, signals), others, 4, 8)
        assert torch.equal(got, want)
    assert encoder._level_signals(index, coords, stride, signals, 7, 4) is None                     # more than there are
    assert encoder._level_signals(index, coords, stride, signals.requires_grad_(), others, 4) is None


@pytest.mark.parametrize("n", [1, 2, 1000])
def test_segments_keys_and_rows_apart(hip_lib, n):
    from swin3d_amd import encoder
    from swin3d_amd.sparse_dl.knn.knn import knn_query
    coords, signals = _level(n, n, 2, 10, batches=3)
    n = coords.shape[0]
    host = coords.cpu()
    for batches in (1, 3, 5, 700):
        assert torch.equal(encoder.segment_offsets(coords[:, 0], batches).cpu(), encoder.segment_offsets(host[:, 0], batches))
    shifted = coords - torch.tensor([0, 40, 0, 7], dtype=torch.int32, device="cuda") * 2
    assert torch.equal(encoder.conv3x3x3_neighbours(shifted, 2).cpu(), encoder.conv3x3x3_neighbours(shifted.cpu(), 2))
    ends = encoder.segment_offsets(coords[:, 0], 3)
    apart = knn_query(3, signals[:, 1:4], signals[:, 1:4], ends, ends, strided=True)
    dense = knn_query(3, signals[:, 1:4].contiguous(), signals[:, 1:4].contiguous(), ends, ends)
    assert torch.equal(apart[0], dense[0]) and torch.equal(apart[1], dense[1])
    if n > 1:
        with pytest.raises(RuntimeError, match="contiguous"):
            knn_query(3, signals[:, 1:4], signals[:, 1:4], ends, ends)


@pytest.mark.parametrize("sizes", [(1, 1), (63, 64), (65, 129), (4096, 4097), (30011, 262_145), (0, 7)])
@pytest.mark.parametrize("batches", [1, 2, 5, 300])
def test_ends_of_two_columns(hip_lib, sizes, batches):
    """Around the sizes where the search takes another step, elements without rows among them, columns of wider rows."""
    from swin3d_amd import encoder
    gen = torch.Generator().manual_seed(sizes[1] + batches)
    columns = [torch.randint(0, max(1, batches - 1), (n, 1 + i), generator=gen, dtype=torch.int32).sort(0)[0].cuda() for i, n in enumerate(sizes)]
    columns = [c[:, -1] for c in columns]
    got = encoder.segment_offsets_of_two(*columns, batches)
    for column, ends in zip(columns, got):
        want = torch.searchsorted(column.cpu().contiguous(), torch.arange(batches, dtype=torch.int32), right=True)
        assert ends.dtype == torch.int32 and torch.equal(ends.cpu().long(), want) and torch.equal(encoder.segment_offsets(column, batches), ends)


def test_ends_of_more_elements_than_a_launch_has_wavefronts(hip_lib):
    """2^26 wavefronts are as many threads as a launch may have."""
    from swin3d_amd import encoder
    count = 2 ** 26 + 12_345
    column = torch.tensor([0, 0, 3, 70_000, 2 ** 26 + 5], dtype=torch.int32, device="cuda")
    ends = encoder.segment_offsets(column, count)
    want = torch.full((count,), 4, dtype=torch.int32, device="cuda")
    want[:3], want[3:70_000], want[2 ** 26 + 5:] = 2, 3, 5
    assert torch.equal(ends, want)


@pytest.mark.parametrize("n,stride", [(1, 1), (7, 1), (8, 2), (9, 3), (4096, 1), (4097, 2), (30011, 1)])
def test_stem_neighbours_in_any_order_and_twice(hip_lib, n, stride):
    """Rows in any order, around the sizes where the table doubles, dense and sparse, some coordinates twice: the first
    row is the one that counts."""
    from swin3d_amd import encoder
    side = max(2, round((2 * n) ** (1 / 3)))
    generator = torch.Generator().manual_seed(n)
    coords = torch.randint(-side // 2, side // 2 + 1, (n, 4), generator=generator, dtype=torch.int32) * stride
    coords[:, 0] = torch.randint(0, 3, (n,), generator=generator, dtype=torch.int32)
    first = {}
    for row, voxel in enumerate(coords.tolist()):
        first.setdefault(tuple(voxel), row)
    offsets = [(x, y, z) for x in (-1, 0, 1) for y in (-1, 0, 1) for z in (-1, 0, 1)]
    want = torch.tensor([[first.get((b, x + dx * stride, y + dy * stride, z + dz * stride), n) for dx, dy, dz in offsets]
                         for b, x, y, z in coords.tolist()])
    assert torch.equal(encoder.conv3x3x3_neighbours(coords.to("cuda"), stride).cpu(), want)


@pytest.mark.parametrize("n,width,dtype", [(1, 1, torch.float16), (19, 3, torch.float32), (1896, 9, torch.float16), (1897, 9, torch.float32),
                                           (500, 6, torch.float16), (60, 257, torch.float16), (7, 1024, torch.float32)])
def test_stem_rows_side_by_side(hip_lib, n, width, dtype):
    """The stem's gather: part of a workgroup's rows, whole ones, rows wider than a workgroup; the row of zeros from either end."""
    from swin3d_amd import encoder
    generator = torch.Generator().manual_seed(n)
    feats = torch.randn(n, width, generator=generator).to(dtype)
    feats[0, 0] = float("inf")
    rows = torch.randint(-n - 1, n + 1, (n, 27), generator=generator)
    want = torch.cat([feats, feats.new_zeros(1, width)])[rows.reshape(-1)].view(n, 27 * width)
    assert torch.equal(encoder._gather_rows(feats.cuda(), rows.cuda()).cpu(), want)
    feats = feats.cuda()
    assert encoder._gather_rows(feats.t().contiguous().t(), rows.cuda()) is None or width == 1 or n == 1
    assert encoder._gather_rows(feats, rows.int().cuda()) is None
    assert encoder._gather_rows(feats.requires_grad_(), rows.cuda()) is None
    outside = rows.cuda()
    outside[0, 0], outside[0, 1] = n + 1, -n - 2       # no such rows
    got = encoder._gather_rows(feats.detach(), outside).view(n * 27, width)
    assert got[:2].isnan().all() and torch.equal(got[2:].cpu(), want.view(n * 27, width)[2:])


@pytest.mark.parametrize("rows", [-1, 1])
def test_rows_that_are_not_the_voxels_own(hip_lib, rows):
    """Fewer or more signal rows than voxels, and signals on the host: no kernel takes them, and a stage refuses them."""
    from swin3d_amd import encoder
    from swin3d_amd.window_index import build_window_indices
    coords, signals = _level(8, 600, 1, 10)
    wrong = signals[:rows] if rows < 0 else torch.cat([signals, signals[:rows]])
    stage = encoder.Stage(48, 2, 6, 5, 4, cRSE="XYZ_RGB_NORM").cuda()
    index = build_window_indices(coords, 1, 2, (0,))[0]
    for s in (wrong, signals.cpu()):
        assert encoder._pool_level(coords, 2, s, index) is None and encoder._level_signals(index, coords, 1, s, 6, 4) is None
        with pytest.raises((ValueError, RuntimeError)):
            stage.plan(coords, 1, s)
    stage.plan(coords, 1, signals)


@pytest.mark.parametrize("how", ["kernel", "tensors"])
def test_a_cell_that_no_point_stands_for(hip_lib, how):
    """NaN among the signals of a cell's points: no member is the nearest to their mean.  The next level says so, on the
    kernel and where tensor operations pool (signals that want a gradient)."""
    from swin3d_amd import encoder
    coords, signals = _level(9, 900, 1, 10)
    stages = [encoder.Stage(48, 1, 6, 5, 4, cRSE="XYZ_RGB_NORM").cuda() for _ in range(2)]
    signals[17, 5] = float("nan")
    signals.requires_grad_(how == "tensors")
    _, (coarse, coarse_signals, _) = stages[0].plan(coords, 1, signals, 2)
    bad = coarse[:, 0] < 0
    assert bad.sum() == 1 and coarse_signals[bad].isnan().all() and not coarse_signals[~bad].isnan().any()
    with pytest.raises(ValueError, match="NaN among their signals"):
        stages[1].plan(coarse, 2, coarse_signals, 2)
    net = encoder.Swin3DEncoder([1, 1], [48, 96], [6, 6], [5, 5], 4, num_layers=2, in_channels=6, cRSE="XYZ_RGB_NORM", fp16_mode=2).cuda()
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16), pytest.raises(ValueError, match="NaN among their signals"):
        net(encoder.SparseVoxels(coords, torch.zeros(900, 6, device="cuda"), 1), signals)

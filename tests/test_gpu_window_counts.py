"""Window sets by the counting sort where their lattice ends at a workgroup's last cell, before and behind it, and the counts
that the host waits for, against the sort of all voxels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [(16, 16, 16), (16, 16, 17), (4095, 1, 1), (4097, 1, 1), (1, 1, 1), (32, 16, 16), (32, 32, 32)])
def test_lattice_edges(hip_lib, monkeypatch, box):
    from swin3d_amd import window_index
    rng = np.random.default_rng(box[0])
    n = max(5000, box[0] * box[1] * box[2] // 2 + 1)
    cells = np.stack([rng.integers(0, e, n) for e in box], 1)
    cells[0], cells[1] = 0, np.array(box) - 1
    coords = torch.from_numpy(np.concatenate([np.zeros((n, 1), np.int64), cells], 1).astype(np.int32)).cuda()
    sets = [(1, 0), (2, 1), (5, 2)]
    by_grid = window_index.build_window_indices(coords, 1, 5, sets)
    monkeypatch.setattr(window_index, "USE_GRID_PATH", False)
    by_sort = window_index.build_window_indices(coords, 1, 5, sets)
    for a, b in zip(by_grid, by_sort):
        assert (a.num_windows, a.num_pairs, a.max_window_voxels) == (b.num_windows, b.num_pairs, b.max_window_voxels)
        for name in ("n2n", "w_w_id", "w_sizes", "w2n"):
            assert torch.equal(getattr(a, name), getattr(b, name)), name


@pytest.mark.parametrize("sets", [[(5, 0)], [(5, 0), (5, 2)], [(2, 0), (5, 0), (5, 2), (7, 3), (10, 4)]])
def test_sets_are_finished_on_return(hip_lib, sets):
    """Nothing of the call is on its way when it returns, so another stream may read the sets without an event."""
    from swin3d_amd import window_index
    rng = np.random.default_rng(4)
    cells = np.unique(rng.integers(0, (400, 400, 6), (400_000, 3)), axis=0).astype(np.int32)
    coords = torch.from_numpy(np.concatenate([np.zeros_like(cells[:, :1]), cells], 1)).cuda()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        built = window_index.build_window_indices(coords, 1, 5, sets)
    assert side.query()
    for got, alone in zip(built, sets):
        again = window_index.window_sets(coords, 1, 5, [alone])[0]
        assert torch.equal(got.n2n, again.n2n) and torch.equal(got.w_sizes, again.w_sizes) and got.num_pairs == again.num_pairs

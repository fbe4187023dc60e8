"""The KNN grid at the edges of its forms (one workgroup, several kernels; groups of four, eight and sixteen lanes; rows of cells
longer than a workgroup takes at a time) against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(oracle_lib, K, src, qry, src_end, qry_end, cell=0.0):
    from swin3d_amd.sparse_dl.knn.knn import knn_query
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    idx, dist2 = knn_query(K, t(src), t(qry), t(np.int32(src_end)), t(np.int32(qry_end)), cell)
    ref_idx, ref_dist2 = oracle_lib.knn(K, src, qry, np.int32(src_end), np.int32(qry_end))
    assert np.array_equal(idx.cpu().numpy(), ref_idx) and np.array_equal(dist2.cpu().numpy(), ref_dist2)


def _surface(rng, n, scale=1.0):
    """points near the faces of a box"""
    p = rng.random((n, 3)).astype(np.float32)
    p[np.arange(n), rng.integers(0, 3, n)] *= np.float32(0.02)
    return p * np.float32(scale)


@pytest.mark.parametrize("ns", [1, 2, 63, 1024, 1025, 4095, 4096, 4097, 20000])
@pytest.mark.parametrize("K", [1, 3, 4, 5, 8, 16, 17])
def test_sizes_and_groups(oracle_lib, hip_lib, ns, K):
    rng = np.random.default_rng(ns + K)
    src, qry = _surface(rng, ns, 7.0), _surface(rng, 300, 7.5)
    third = ns // 3
    _check(oracle_lib, K, src, qry, [third, ns], [100, 300])


@pytest.mark.parametrize("ns", [700, 5000])
@pytest.mark.parametrize("nq", [65536, 65537, 200001])    # groups of sixteen, of four
def test_many_queries(oracle_lib, hip_lib, ns, nq):
    rng = np.random.default_rng(nq)
    _check(oracle_lib, 3, _surface(rng, ns), _surface(rng, nq), [ns], [nq])


@pytest.mark.parametrize("ns", [300, 4096, 12000])
def test_sources_on_a_line(oracle_lib, hip_lib, ns):
    """One row of cells, longer than a workgroup takes at a time; sources behind the last segment are no one's."""
    rng = np.random.default_rng(ns)
    src = np.zeros((ns, 3), np.float32)
    src[:, 0] = rng.random(ns) * 1000
    qry = np.zeros((200, 3), np.float32)
    qry[:, 0] = rng.random(200) * 1000
    for cell in (0.0, 0.05, 5000.0):
        _check(oracle_lib, 4, src, qry, [ns - ns // 10], [200], cell)


@pytest.mark.parametrize("ns", [100, 9000])
def test_many_segments(oracle_lib, hip_lib, ns):
    rng = np.random.default_rng(ns)
    ends = np.sort(rng.integers(0, ns, 63))
    _check(oracle_lib, 3, _surface(rng, ns), _surface(rng, 640), [*ends, ns], np.arange(10, 650, 10))

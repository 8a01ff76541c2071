"""Delaunay triangulation at the sizes where its rounds change: lists of
changed triangles that one workgroup takes, scans of one and of three
launches, bids in LDS or memory, and the point count from which points are
kept in Z order, with duplicates and constraints there.  Compared with
scipy.spatial.Delaunay (Qhull) on points in general position."""
import numpy as np
import pytest
from scipy.spatial import Delaunay as Qhull

from test_gpu_delaunay import tri_set

pytestmark = pytest.mark.gpu


def points(n, seed):
    return np.random.default_rng(seed).random((n, 2)) * 1000.0


@pytest.mark.parametrize("n", [3, 4, 341, 683, 1025, 2046, 2047, 2048, 4095, 8191, 16383, 16385,
                               65535, 65536, 65537])
def test_equals_scipy_at_the_edges(gpu, n):
    from cvtamd.delaunay import delaunay
    p = points(n, n)
    tri, opp = delaunay(p)
    assert tri_set(tri) == tri_set(Qhull(p).simplices)


@pytest.mark.parametrize("n", [65000, 65530])
def test_duplicates_on_either_side_of_the_order(gpu, n):
    from cvtamd.delaunay import Delaunay
    p = points(n, 7)
    g = np.random.default_rng(8)
    both = np.concatenate([p, p[g.integers(0, n, 600)]])[g.permutation(n + 600)]
    uniq, inv = np.unique(both, axis=0, return_inverse=True)
    with Delaunay(len(both)) as d:
        tri, _ = d.compute(both)
        assert d.stats()["duplicates"] == 600
        again, _ = d.compute(p)                   # the context after another order
    assert tri_set(inv.reshape(-1)[tri]) == tri_set(Qhull(uniq).simplices)
    assert tri_set(again) == tri_set(Qhull(p).simplices)


@pytest.mark.parametrize("n", [65400, 65700])
def test_constraints_on_either_side_of_the_order(gpu, n):
    from cvtamd.delaunay import delaunay
    k = 64
    a = 2 * np.pi * (np.arange(k) + 0.25) / k
    ring = np.stack([500 + 300 * np.cos(a), 500 + 300 * np.sin(a)], 1)
    p = points(n - k, 9)
    p = p[np.abs(np.hypot(*(p - 500).T) - 300) > 1.0]
    pts = np.concatenate([p, ring])
    segs = np.stack([len(p) + np.arange(k), len(p) + (np.arange(k) + 1) % k], 1).astype(np.int32)
    tri, opp = delaunay(pts, segments=segs)
    edges = np.sort(np.concatenate([tri[:, [0, 1]], tri[:, [1, 2]], tri[:, [2, 0]]]), axis=1)
    have = set(map(tuple, edges.tolist()))
    assert all(tuple(sorted(s)) in have for s in segs.tolist())
    marked = ((opp >= 0) & ((opp & 4) != 0)).sum()
    assert marked == 2 * k

"""Prefix sums on both sides of the sizes where their launches change: 4096,
8192, 16384 and 24576 counts in one workgroup, three launches beyond (for the
triangulation's bids from 8193 on), reached through the calls that scan them.
Bar: bit-exact, and the unique triangulation."""
import numpy as np
import pytest
from scipy.spatial import Delaunay as Qhull

from test_gpu_delaunay import tri_set

pytestmark = pytest.mark.gpu

EDGES = [4096, 8192, 16384, 24576, 32768]


def fan_mesh(nv, seed):
    """nv vertices in a strip of triangles, shuffled"""
    g = np.random.default_rng(seed)
    i = np.arange(nv)
    uv = np.stack([i // 2 + 0.3 * g.random(nv), (i % 2) + 0.3 * g.random(nv)], 1)
    p3 = np.stack([uv[:, 0], uv[:, 1], np.sin(0.1 * uv[:, 0])], 1)
    tri = np.stack([i[:-2], i[1:-1], i[2:]], 1).astype(np.int32)
    return uv, p3, tri[g.permutation(len(tri))]


@pytest.mark.parametrize("nv", [e + d for e in EDGES for d in (-1, 0, 1, 3)])
def test_vertex_weights(gpu, orc, nv):
    from cvtamd.weighting import vertex_weights
    uv, p3, tri = fan_mesh(nv, nv)
    assert np.array_equal(vertex_weights(uv, p3, tri), orc.vertex_weights(uv, p3, tri))


@pytest.mark.parametrize("side", [90, 91, 128, 129, 156, 157, 181, 182])   # squared: the tiles
def test_raster(gpu, orc, side):
    from cvtamd import compat
    n = 16 * side - 5
    g = np.random.default_rng(side)
    uv, _, tri = fan_mesh(60, side)
    uv = (uv - uv.min(0)) / (uv.max(0) - uv.min(0)).max()
    w = g.random(len(uv))
    scale = 1.0 / (n - 1)
    assert np.array_equal(compat.rasterize(uv, w, tri, scale, n), orc.raster(uv, w, tri, scale, n))


# 2 n - 2 triangles at the end, infinite ones included
@pytest.mark.parametrize("n", [e // 2 + d for e in EDGES for d in (0, 1, 2)])
def test_delaunay(gpu, n):
    from cvtamd.delaunay import delaunay
    p = np.random.default_rng(n).random((n, 2)) * 1000.0
    tri, _ = delaunay(p)
    assert tri_set(tri) == tri_set(Qhull(p).simplices)

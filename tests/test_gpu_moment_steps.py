"""Moments on both sides of the rule by which a wave's loads run ahead and its
record queue is carried over its steps (csrc/cvt_kernels.h).  Densities are
whole numbers up to 4 and sites lie on pixel centres, so every partial sum is
a whole number below 2^24 and the oracle's fp64 sums are exact as well: the
moments are equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,S,tile", [
    (2048, 1536, 12000, 64),    # 768 tiles, the most that run ahead
    (2048, 1537, 12000, 64),    # 800 tiles, the last row of them one pixel high
    (515, 387, 8000, 64),       # 25 pixels per site: the queue fills within a step; ragged tiles
    (1000, 900, 900, 128),      # eight steps per wave, records of all of them in one drain
    (4096, 2304, 9000, 128),    # 576 tiles of 128
    (4096, 3200, 9000, 128),    # 800 tiles of 128
    (40, 3, 20, 64),            # steps without rows, fewer steps than waves
])
def test_moments_equal_oracle(gpu, orc, W, H, S, tile):
    import cvtamd
    g = np.random.default_rng(W + H + S)
    at = g.choice(W * H, S, replace=False)
    xy = (np.stack([at % W, at // W], 1) + 0.5).astype(np.float32)
    rho = g.integers(0, 5, (H, W)).astype(np.float32)
    rho[0, 0] = 4.0
    with cvtamd.Engine(W, H, S) as e:
        e.set_density(rho)
        e.tile = tile
        e.set_sites(xy)
        e.voronoi()
        lab = e.labels()
        m = e.moments()
    assert np.array_equal(m, orc.moments(rho, lab, xy))

"""The dense JFA passes on grids whose width is no multiple of four and that
are large enough for runs of rows (the row's last quad overlaps the one before
it, and its right taps can cross the row's end by one to three pixels): the
label map equals the oracle's JFA bit for bit."""
import numpy as np
import pytest

from test_gpu_jfa_lattice import labels, random_sites

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,S", [
    (1025, 3001, 1500),     # one pixel in the last segment; the 16 KB table
    (2049, 2051, 30000),    # first step 2048, taken partly by the last quad; split table
    (2050, 1500, 12000),    # two pixels over, the 160 KB table
    (2051, 1300, 2048),     # three over, the smallest 40 KB table
    (1279, 2999, 18000),    # one pixel short of whole segments
    (4099, 800, 20000),     # wide: first step 4096, left taps partly off the grid at no lane
    (517, 7001, 9000),      # five pixels in the last segment, few segments
    (765, 512, 18000),      # the fewest runs that are taken (1.5 per CU), a table of 160 KB
    (67, 8191, 900),        # step 64 (of the row's last quad) between W - 4 and W
    (9, 8191, 300),         # the smallest width
    (2049, 2051, 140000),   # more than eight sites per class of the first passes: every step dense,
                            # step 2048 between W - 4 and W
    (1025, 1024, 40000),
])
def test_labels_equal_oracle(gpu, orc, W, H, S):
    xy = random_sites(W + H + S, W, H, S)
    assert np.array_equal(labels(W, H, xy), orc.jfa(W, H, xy))


@pytest.mark.parametrize("W,H,S", [(9, 12, 5), (11, 70, 40), (13, 40, 20), (98, 77, 150),
                                   (259, 130, 5000), (67, 300, 30000)])
def test_forced_runs_equal_oracle(gpu, orc, W, H, S):
    """runs asked for at every step, on grids of any size"""
    import cvtamd
    xy = random_sites(W + H + S, W, H, S)
    with cvtamd.Engine(W, H, S) as e:
        e.jfa_shape = (1 << 13) - 1, 0
        e.set_sites(xy)
        e.voronoi()
        lab = e.labels()
    assert np.array_equal(lab, orc.jfa(W, H, xy))

"""The dense JFA passes with a site table beyond LDS on whole 256-pixel
segments (a lane's neighbour sites read across the wave): the label map
equals the oracle's JFA bit for bit."""
import numpy as np
import pytest

from test_gpu_jfa_lattice import labels, random_sites

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,S", [
    (512, 8191, 30000),      # two segments, each at an edge of the grid; ragged chains of rows
    (768, 5500, 21000),      # three segments
    (2304, 1900, 20479),     # nine segments, the smallest table beyond LDS
    (2048, 2048, 60000),     # too dense for the lattice passes: steps 128 and up as well
])
def test_labels_equal_oracle(gpu, orc, W, H, S):
    xy = random_sites(W + H + S, W, H, S)
    assert np.array_equal(labels(W, H, xy), orc.jfa(W, H, xy))

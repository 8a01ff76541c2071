"""The first five JFA passes on residue classes (csrc/jfa_lattice.hip): the
label map equals the oracle's JFA bit for bit at the edges of the launch's
rule and of its mask path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def labels(W, H, xy):
    import cvtamd
    with cvtamd.Engine(W, H, len(xy)) as e:
        e.set_sites(xy)
        e.voronoi()
        return e.labels()


def random_sites(seed, W, H, S):
    g = np.random.default_rng(seed)
    return (g.random((S, 2)) * [W, H]).astype(np.float32)


@pytest.mark.parametrize("W,H,S", [
    (65, 65, 20),        # the smallest first step (64) that takes it
    (128, 33, 20),       # the shortest side it takes, one lattice row of some classes
    (129, 128, 80),      # a first step of 128 with one column beyond it
    (255, 257, 300),     # odd in both sides, the last row and column ragged
    (513, 300, 700),     # first step 512 on a grid barely above it
    (1022, 768, 3900),   # width 2 mod 4 near the rule's 200 pixels per site
    (2048, 1030, 10000), # sixteen-wave groups, ragged rows
    (4096, 2051, 9000),  # eight-wave groups
    (512, 512, 1),       # one site
    (512, 512, 2048),    # eight sites per class, the most that take it; dense classes likely
    (1024, 1024, 8192),
    (1100, 700, 32768),  # the same on classes of 18 x 11 points
    (2048, 2048, 32768),
    (2047, 2048, 32769), # one site too many
])
def test_labels_equal_oracle(gpu, orc, W, H, S):
    xy = random_sites(W + H + S, W, H, S)
    assert np.array_equal(labels(W, H, xy), orc.jfa(W, H, xy))


@pytest.mark.parametrize("n,per", [(512, 16), (512, 17), (512, 18), (2048, 17), (1024, 400)])
def test_classes_at_and_past_the_mask_capacity(gpu, orc, n, per):
    """`per` seeds in one residue class (16 fit a wave's masks; with 17 and
    more the class takes the dense evaluation), the rest spread"""
    first = 1 << ((n - 1).bit_length() - 1)
    s = first // 16
    g = np.random.default_rng(per)
    cell = g.choice((n // s) ** 2, per, replace=False)
    # pixels (5 mod s, 3 mod s), in a random label order
    one = np.stack([s * (cell % (n // s)) + 5.5, s * (cell // (n // s)) + 3.25], 1)
    xy = np.concatenate([one, g.random((n * n // 400, 2)) * n]).astype(np.float32)
    xy = xy[g.permutation(len(xy))]
    assert np.array_equal(labels(n, n, xy), orc.jfa(n, n, xy))


def test_shared_pixels_ties_and_off_grid_sites(gpu, orc):
    """equal sites, sites sharing a pixel, exact distance ties (sites on pixel
    corners of a coarse grid) and sites off the grid"""
    n = 256
    a = np.arange(8, n, 32, dtype=np.float32)
    grid = np.stack(np.meshgrid(a, a), -1).reshape(-1, 2)
    xy = np.concatenate([grid, grid[::3], grid[::5] + np.float32(0.5),
                         np.array([[-40, 30], [300, 300], [10, -200], [256, 256]], np.float32)])
    xy = xy[np.random.default_rng(1).permutation(len(xy))].astype(np.float32)
    assert np.array_equal(labels(n, n, xy), orc.jfa(n, n, xy))


def test_site_counts_on_either_side_of_the_rule(gpu, orc):
    """one engine, site sets that take the lattice launch, the seed scatter
    and the lattice launch again: the maps the two keep between runs agree"""
    import cvtamd
    n = 256
    with cvtamd.Engine(n, n, 4000) as e:
        e.set_density(np.ones((n, n), np.float32))
        for S in (300, 4000, 200, 330, 2000):
            xy = random_sites(S, n, n, S)
            e.set_sites(xy)
            e.voronoi()
            assert np.array_equal(e.labels(), orc.jfa(n, n, xy)), S
            e.lloyd_until(9, target=1e30)
            e.lloyd(3)
            e.voronoi()
            assert np.array_equal(e.labels(), orc.jfa(n, n, e.sites())), S


def test_batch_of_patches_on_both_sides_of_the_rule(gpu, orc):
    """patches with and without the lattice launch in one batch (first steps of
    32 .. 1024, ragged sides, dense and sparse sites), then other site counts
    that swap them"""
    import cvtamd
    sizes = [(64, 64), (128, 100), (132, 150), (260, 300), (520, 512), (1100, 700), (300, 256)]
    few = [20, 60, 90, 350, 1200, 3500, 3000]
    many = [20, 60, 700, 3500, 1200, 3800, 300]
    with cvtamd.Batch(sizes, [max(a, b) for a, b in zip(few, many)]) as b:
        for counts in (few, many, few):
            xys = [random_sites(k + n, w, h, n) for k, ((w, h), n) in enumerate(zip(sizes, counts))]
            for k, ((w, h), xy) in enumerate(zip(sizes, xys)):
                b.set_density(k, np.ones((h, w), np.float32))
                b.set_sites(k, xy)
            b.voronoi()
            for k, ((w, h), xy) in enumerate(zip(sizes, xys)):
                assert np.array_equal(b.labels(k), orc.jfa(w, h, xy)), (counts, k)
            b.lloyd(2)
            b.voronoi()
            for k, (w, h) in enumerate(sizes):
                assert np.array_equal(b.labels(k), orc.jfa(w, h, b.sites(k))), (counts, k)


@pytest.mark.parametrize("W,H,S", [
    (65, 70, 2000),      # no lattice launch: dense passes, then five fused
    (130, 129, 90),      # lattice, then the last four fused
    (127, 66, 40),       # lattice, then the last three fused
    (301, 33, 2047),     # the largest 16 KB table
    (517, 260, 2048),    # the smallest 40 KB table
    (1021, 530, 5118),   # the largest 40 KB table
    (1021, 530, 5119),   # too large for the fused passes
])
def test_fused_tail_at_widths_not_a_multiple_of_four(gpu, orc, W, H, S):
    xy = random_sites(7 * W + S, W, H, S)
    assert np.array_equal(labels(W, H, xy), orc.jfa(W, H, xy))

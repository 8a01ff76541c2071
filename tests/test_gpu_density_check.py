"""The density check on the device (k_density_max): refused values wherever
they lie, accepted edge values, and the power-of-two scale it gives (energies
equal the oracle's)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 72


@pytest.mark.parametrize("where", [0, 1023, 1024, N * N - 1])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, -1.0, np.float32(-1e-45)])
def test_bad_values_are_refused(gpu, value, where):
    import cvtamd
    rho = np.ones(N * N, np.float32)
    rho[where] = value
    rho = rho.reshape(N, N)
    with cvtamd.Engine(N, N, 4) as e, cvtamd.Batch([(N, N)], [4]) as b:
        with pytest.raises(cvtamd.CvtError, match="ERR_ARG"):
            e.set_density(rho)
        with pytest.raises(cvtamd.CvtError, match="ERR_ARG"):
            b.set_density(0, rho)
        # a good density afterwards is taken
        e.set_density(np.ones((N, N), np.float32))
        b.set_density(0, np.ones((N, N), np.float32))


@pytest.mark.parametrize("scale", [0.0, -0.0, 1.0, 3e-3, 1.5e30])
def test_scales(gpu, orc, scale):
    """engine and batch agree bit for bit, also when the density's scale
    changes on a context that has run, and match the oracle's energies"""
    import cvtamd
    g = np.random.default_rng(3)
    xy = (g.random((40, 2)) * N).astype(np.float32)
    first = g.random((N, N)).astype(np.float32)
    rho = (g.random((N, N)) * scale).astype(np.float32)
    with cvtamd.Engine(N, N, 40) as e, cvtamd.Batch([(N, N)], [40]) as b:
        e.tile = b.tile(0)
        for r in (first, rho):
            e.set_density(r)
            e.set_sites(xy)
            e.clear_history()
            e.lloyd(3)
            b.set_density(0, r)
            b.set_sites(0, xy)
            b.set_tile(0, e.tile)
            b.lloyd(3)
            b.synchronize()
        h = e.history()
        assert np.array_equal(e.sites(), b.sites(0))
        assert np.array_equal(h, b.history(0)[3:])
    if scale > 1e-30:
        _, ref, _ = orc.lloyd(rho, xy, 3)
        assert np.allclose(h[:, 0], ref, rtol=1e-5)
    elif scale == 0.0:
        assert np.all(h == 0.0)

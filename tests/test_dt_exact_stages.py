"""The exact stages of the triangulation's predicates (wrapping 64- and 128-bit
integers, then the wide evaluation; dt_predicates.h) against rational
arithmetic and the symbolic perturbation, on degenerate and nearly degenerate
records whose finest bit lies 2^0 .. 2^-60 below the coordinates' size, so that
every stage and both sides of its limits decide some of them."""
import numpy as np
import pytest

from dt_cases import degenerate_records, exact_incircle, exact_orient, sos_incircle, sos_orient
from test_dt_predicates import PERMS, harness  # noqa: F401


def fine_records(j, scale, seed):
    """degenerate records times `scale`, moved by a multiple of 2^-j that keeps
    them exact, and the same with one coordinate 2^-j off"""
    g = np.random.default_rng(seed)
    q = degenerate_records(seed)
    q = q[g.choice(len(q), 24, replace=False)] * scale
    step = 2.0 ** -j
    off = np.floor(g.random((len(q), 2)) * 1000.0) * step
    moved = q + np.tile(off, 4)
    exact = np.all(moved - np.tile(off, 4) == q, axis=1)
    near = q.copy()
    k = g.integers(0, 8, len(q))
    near[np.arange(len(q)), k] += np.where(g.random(len(q)) < 0.5, step, -step)
    return np.concatenate([q, moved[exact], near])


@pytest.mark.parametrize("scale", [1.0, 0.5, 2.0 ** -40, 2.0 ** 30])
@pytest.mark.parametrize("j", [0, 6, 10, 13, 16, 20, 24, 28, 32, 36, 40, 44, 52, 60])
def test_signs_at_every_stage(harness, j, scale):  # noqa: F811
    # the finest bit relative to the scaled coordinates
    q = fine_records(j - int(np.log2(scale)), scale, j)
    got = harness(q)
    assert (got[:, 2] == 0).all()
    for i, r in enumerate(q):
        o, c = exact_orient(r), exact_incircle(r)
        assert got[i, 0] == o and got[i, 1] == c, (i, r)
        idx = PERMS[i % 6]
        assert got[i, 3] == (o if o else sos_orient(r, idx[:3])), (i, r)
        assert got[i, 4] == (c if c else sos_incircle(r, idx)), (i, r)

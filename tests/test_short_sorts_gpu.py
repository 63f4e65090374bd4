"""Sorts on both sides of the line between counting and digit passes.  The gradient's slots
(four per constraint) are sorted by vertex, keys of two digits, by counting up to 3,200 of
them and by digits beyond; slots of one vertex keep their order, so the sums have one order.

Bar: 1e-11 of the largest entry against the oracle, as for whole sets; two calls give the
same bits."""
import numpy as np
import pytest

import oracle as O
from cipc import Simulator, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def state(require_gpu):
    sd = scenes.cloth_on_sphere(sheets=3, n=18, y0=0.2008, dy=0.0008, sphere_level=1, seed=2, twists=[0.0, 5.0, 10.0])
    sd.X[:sd.n_cloth, 0] *= 0.03 * 18 / 14
    sd.X[:sd.n_cloth, 2] *= 0.03 * 18 / 14
    sim, orc = Simulator(sd), O.OracleScene(sd, threads=2)
    x = sd.X.ravel().copy()
    C = orc.constraint_set(x)
    assert len(C) > 6000 and sd.nV + 1 > 512     # two digits
    yield sim, orc, x, np.ascontiguousarray(C[np.random.default_rng(1).permutation(len(C))])
    sim.close()


@pytest.mark.parametrize("n", [1, 799, 800, 801, 1250, 6000])
def test_gradient_of_sets_around_the_line(state, n):
    sim, orc, x, C = state
    kappa = orc.scalars()["kappa"]
    sub = np.ascontiguousarray(C[:n])
    g, go = sim.barrier_gradient(x, sub, kappa), orc.gradient(x, sub, kappa)[1]
    assert np.abs(g - go).max() <= 1e-11 * np.abs(go).max()
    assert np.array_equal(g, sim.barrier_gradient(x, sub, kappa))

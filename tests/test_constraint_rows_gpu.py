"""Constraint sets as the caller holds them (int4 rows) on both sides of the line between the
host's and the device's transposition to the library's layout, 16,384 rows, and an empty set.

Bar: distances the same bits as the oracle's, energy 1e-11 (order of the sum), as elsewhere."""
import numpy as np
import pytest

import oracle as O
from cipc import Simulator, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def state(require_gpu):
    sd = scenes.cloth_on_sphere(sheets=3, n=30, y0=0.2008, dy=0.0008, sphere_level=1, seed=2, twists=[0.0, 5.0, 10.0])
    sd.X[:sd.n_cloth, 0] *= 0.03 * 30 / 14
    sd.X[:sd.n_cloth, 2] *= 0.03 * 30 / 14
    sim, orc = Simulator(sd), O.OracleScene(sd, threads=2)
    x = sd.X.ravel().copy()
    C = orc.constraint_set(x)
    assert len(C) > 17000
    yield sim, orc, x, C
    sim.close()


@pytest.mark.parametrize("n", [0, 1, 3, 16383, 16384, 16385, 17000])
def test_distances_and_energy_of_n_rows(state, n):
    sim, orc, x, C = state
    sub = np.ascontiguousarray(C[:n])
    kappa = orc.scalars()["kappa"]
    e, eo = sim.barrier_energy(x, sub, kappa), orc.energy(x, None, sub, kappa)[0][3]
    assert abs(e - eo) <= 1e-11 * abs(eo)
    if n:
        d, least = sim.min_dist2(x, sub)
        do = orc.dist2_list(x, sub)
        assert np.array_equal(d, do) and least == do.min()

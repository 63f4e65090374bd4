"""Candidate walk of the broad phases at the sizes where it can go wrong: fewer items than
one workgroup takes, query boxes of one cell and of more cells than an item has lanes, cells
with more records than one pass, more large primitives than one pass reads, none at all.

The constraint set is bit-exact against the oracle's for every cell size (the grid only
chooses the candidates); the CCD step equals the oracle's to the parity bar."""
import numpy as np
import pytest

import oracle as O
from cipc import Simulator, scenes

pytestmark = pytest.mark.gpu


def scene(name):
    if name == "tiny":         # 4 cloth vertices, an icosahedron and the ground
        return scenes.cloth_on_sphere(sheets=1, n=2, y0=0.2006, sphere_level=0, seed=1)
    if name == "dense":        # three 3 cm sheets inside d_hat of each other: crowded cells
        sd = scenes.cloth_on_sphere(sheets=3, n=14, y0=0.2008, dy=0.0008, sphere_level=1, seed=2, twists=[0.0, 5.0, 10.0])
        sd.X[:sd.n_cloth, 0] *= 0.03
        sd.X[:sd.n_cloth, 2] *= 0.03
        return sd
    if name == "ground":       # the ground's primitives are large against the sheet's cells
        return scenes.scene_cloth_on_ground(n=13)
    return scenes.scene_codim_contact()


@pytest.mark.parametrize("name", ["tiny", "dense", "ground", "codim"])
@pytest.mark.parametrize("cell", [0.25, 1.0, 4.0])
def test_constraint_set_equals_oracle_for_every_cell_size(require_gpu, name, cell):
    sd = scene(name)
    sim = Simulator(sd)
    sim.set_tuning(cell_mult=cell)
    orc = O.OracleScene(sd, threads=2)
    rng = np.random.default_rng(3)
    for k in range(2):
        x = sd.X.ravel() + (0 if k == 0 else 5e-5 * rng.standard_normal(sd.X.size))
        assert np.array_equal(sim.constraint_set(x), orc.constraint_set(x))
    sim.close()


# short sets are sorted by counting and long ones by digits, short runs of cells are summed
# by one workgroup: 4,600 to 25,000 constraints lie on both sides of both lines
@pytest.mark.parametrize("n", [14, 18, 20, 30])
def test_constraint_set_order_below_and_above_the_short_sorts(require_gpu, n):
    sd = scenes.cloth_on_sphere(sheets=3, n=n, y0=0.2008, dy=0.0008, sphere_level=1, seed=2, twists=[0.0, 5.0, 10.0])
    sd.X[:sd.n_cloth, 0] *= 0.03 * n / 14
    sd.X[:sd.n_cloth, 2] *= 0.03 * n / 14
    sim = Simulator(sd)
    got = sim.constraint_set(sd.X.ravel())
    sim.close()
    assert np.array_equal(got, O.OracleScene(sd, threads=2).constraint_set(sd.X.ravel()))


@pytest.mark.parametrize("name", ["tiny", "dense", "ground", "codim"])
def test_ccd_step_equals_oracle(require_gpu, name):
    sd = scene(name)
    sim = Simulator(sd)
    orc = O.OracleScene(sd, threads=2)
    rng = np.random.default_rng(4)
    for size in (1e-5, 1e-3, 2e-2):
        p = size * rng.standard_normal(sd.X.shape)
        p[sd.dbc_idx] = 0
        a, clamp = sim.ccd_stepsize(sd.X.ravel(), p.ravel())
        b, oclamp = orc.ccd(sd.X.ravel(), p.ravel())
        assert clamp == oclamp
        assert b * (1 - 1e-9) <= a <= b * (1 + 1e-12)
    sim.close()

"""Local barrier Hessians at the sizes where their kernel can go wrong: sets that do not fill
a workgroup or leave one constraint over, every kind of constraint (the mollified ones
included), constraints that are not evaluated (closer than the thickness allows), and runs of
one block's summands that cross a wave of the sum.  A large set goes first, so that blocks
left unwritten would hold its values.

Bar: relative 1e-9 against the oracle's Householder-QL projection, as for whole sets."""
import numpy as np
import pytest

import oracle as O
from cipc import Simulator, scenes

pytestmark = pytest.mark.gpu


def kinds(C):
    edge = np.where((C[:, 2] >= 0) & (C[:, 3] >= 0), 0, np.where(C[:, 3] >= 0, 1, np.where(C[:, 2] >= 0, 2, 3)))
    return np.where(C[:, 0] >= 0, edge, np.where(C[:, 3] >= 0, 4, np.where(C[:, 2] >= 0, 5, 6)))


@pytest.fixture(scope="module")
def state(require_gpu):
    sd = scenes.scene_codim_contact()
    sim, orc = Simulator(sd), O.OracleScene(sd, threads=2)
    x = sd.X.ravel() + 2e-4 * np.random.default_rng(1).standard_normal(sd.X.size)
    C = np.concatenate([orc.constraint_set(sd.X.ravel()), orc.constraint_set(x)])
    assert set(kinds(C)) >= {0, 2, 3, 4, 5, 6}
    yield sim, orc, x, C, orc.scalars()["kappa"]
    sim.close()


def check(sim, orc, x, C, kappa):
    none = np.zeros((0, 4), np.int32)
    D = (orc.hessian(x, C, kappa, which=2) - orc.hessian(x, none, kappa, which=0)).toarray()
    G = sim.hessian(x, C, kappa, which=2).toarray()
    assert np.abs(G - D).max() <= 1e-9 * max(np.abs(D).max(), 1e-300)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 500])
def test_sets_of_any_length(state, n):
    sim, orc, x, C, kappa = state
    sim.hessian(x, C, kappa, which=2)
    check(sim, orc, x, np.ascontiguousarray(C[:n]), kappa)


@pytest.mark.parametrize("kind", [0, 2, 3, 4, 5, 6])
def test_one_kind_at_a_time(state, kind):
    sim, orc, x, C, kappa = state
    sim.hessian(x, C, kappa, which=2)
    check(sim, orc, x, np.ascontiguousarray(C[kinds(C) == kind]), kappa)


def test_long_runs_of_one_block(state):
    sim, orc, x, C, kappa = state
    check(sim, orc, x, np.ascontiguousarray(np.repeat(C[:40], 25, axis=0)), kappa)


@pytest.mark.parametrize("spread", [0.0, 1e-5, 1e-4])
def test_mollified_parallel_edges(require_gpu, spread):
    """two grids one above the other: all edge pairs parallel (spread 0) or nearly so"""
    sd = scenes.cloth_on_sphere(sheets=2, n=6, y0=0.2008, dy=0.0008, sphere_level=0, seed=2, twists=[0.0, 0.0])
    sd.X[:sd.n_cloth, 0] *= 0.05
    sd.X[:sd.n_cloth, 2] *= 0.05
    sim, orc = Simulator(sd), O.OracleScene(sd, threads=2)
    x = sd.X.ravel() + spread * np.random.default_rng(1).standard_normal(sd.X.size)
    C = orc.constraint_set(x)
    check(sim, orc, x, C, orc.scalars()["kappa"])
    sim.close()

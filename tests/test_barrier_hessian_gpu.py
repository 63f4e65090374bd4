"""Local barrier Hessians at the sizes where their kernel can go wrong: sets that do not fill
a workgroup or leave one constraint over, every kind of constraint alone (the three mollified
ones included), constraints that are not evaluated (closer than the thickness allows), and runs
of one block's summands that cross a wave of the sum.  A large set goes first, so that blocks
left unwritten would hold its values.

Bars: whole sets relative 1e-9 against the oracle's Householder-QL projection, as elsewhere.
One constraint at a time, 5e-13 of its own block in Frobenius norm: the rotations stop at an
off-diagonal rest of 1e-13 of the matrix, and the positive part moves by no more than what was
left out (it is the projection onto a convex cone); their own rounding, 36 rotations in some
5 sweeps of 2^-53, is an order below.  The rest of the bar is for the two ways in which kernel
and oracle form the matrix before the projection; measured 1.7e-13 at most."""
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
    assert set(kinds(C)) >= {2, 3}
    check(sim, orc, x, C, orc.scalars()["kappa"])
    sim.close()


def crossing_edges(sd, rng, count):
    """positions and mollified edge-edge rows: pairs of edges at their rest lengths that cross
    at their middles under 0.1 to 1.7 degrees (the mollifier ends at 1.8), 0.2 to 0.9 d_hat
    apart, turned at random"""
    T, X = sd.tris, sd.X
    own = set()
    edges = []
    for e in T[:, :2]:
        if not own & set(e.tolist()):
            own |= set(e.tolist())
            edges.append(e)
    x, rows = X.copy(), []
    for k in range(count):
        (a0, a1), (b0, b1) = edges[2 * k], edges[2 * k + 1]
        Q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        t, gap = rng.uniform(0.002, 0.03), rng.uniform(0.2, 0.9) * sd.params["dHat"]
        la, lb = np.linalg.norm(X[a1] - X[a0]), np.linalg.norm(X[b1] - X[b0])
        c = rng.uniform(-1, 1, 3)
        for v, s, u, h in ((a0, -la / 2, 0.0, 0.0), (a1, la / 2, 0.0, 0.0), (b0, -lb / 2, t, gap), (b1, lb / 2, t, gap)):
            x[v] = c + Q @ np.array([s * np.cos(u), s * np.sin(u), h])
        rows.append((a0, a1, -b0 - 1, b1))
    return x.ravel(), np.array(rows, np.int32)


def check_alone(sim, orc, x, C, kappa, label):
    none = np.zeros((0, 4), np.int32)
    base = orc.hessian(x, none, kappa, which=0)
    worst, filled = 0.0, 0
    for i in range(len(C)):
        row = np.ascontiguousarray(C[i:i + 1])
        D = (orc.hessian(x, row, kappa, which=2) - base).tocsr()
        norm = np.sqrt(D.power(2).sum())
        if norm > 0:      # stencils of Dirichlet vertices alone are projected out
            worst = max(worst, np.sqrt((sim.hessian(x, row, kappa, which=2).tocsr() - D).power(2).sum()) / norm)
            filled += 1
    print("%s: %d constraints, largest error %.1e" % (label, filled, worst))
    assert filled and worst <= 5e-13


@pytest.mark.parametrize("scale", [1.0, 1e5, 1e12])
@pytest.mark.parametrize("kind", [0, 2, 3, 4, 5, 6])
def test_every_constraint_against_its_own_block(state, kind, scale):
    sim, orc, x, C, kappa = state
    sub = C[kinds(C) == kind]
    check_alone(sim, orc, x, sub[:40], scale * kappa, "kind %d, stiffness x %g" % (kind, scale))


@pytest.mark.parametrize("scale", [1.0, 1e5, 1e12])
def test_mollified_edge_edge(require_gpu, scale):
    sd = scenes.cloth_on_sphere(sheets=1, n=24, y0=0.21, sphere_level=0, seed=5)
    sim, orc = Simulator(sd), O.OracleScene(sd, threads=2)
    x, C = crossing_edges(sd, np.random.default_rng(7), 60)
    assert (kinds(C) == 1).all()
    kappa = scale * orc.scalars()["kappa"]
    check(sim, orc, x, C, kappa)
    check_alone(sim, orc, x, C, kappa, "mollified edge-edge, stiffness x %g" % scale)
    sim.close()

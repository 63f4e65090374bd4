"""PCG launch shapes and sizes: every lane / unroll shape of the row loop, systems smaller
than one row group and with ragged last groups, empty and dense contact rows.

Bar: the FP64 residual of the library's own assembled matrix, computed in scipy, is at most
2x the solve's tolerance (the factor covers the rounding of the residual itself), and two
solves of one system give the same bits."""
import numpy as np
import pytest

from cipc import Simulator, scenes

pytestmark = pytest.mark.gpu


def system(n, sheets):
    sd = scenes.cloth_on_sphere(sheets=sheets, n=n, y0=0.2008, dy=0.0008, sphere_level=1, seed=n,
                                twists=[5.0 * k for k in range(sheets)])
    b = np.random.default_rng(n).standard_normal((sd.nV, 3))
    b[sd.dbc_idx] = 0
    return sd, sd.X.ravel().copy(), b.ravel()


@pytest.mark.parametrize("n,sheets", [(2, 1), (5, 1), (9, 3), (17, 2)])
@pytest.mark.parametrize("precision", ["fp64", "mixed", "fp32"])
def test_block_jacobi_shapes(require_gpu, n, sheets, precision):
    sd, x, b = system(n, sheets)
    sim = Simulator(sd, precision=precision)
    C, kappa = sim.constraint_set(x), sim.scalars()["kappa"]
    H = sim.hessian(x, C, kappa)
    for lanes in (4, 8, 16):
        for unroll in (1, 2):
            sim.set_tuning(spmv_grid=1024, spmv_lanes=lanes, spmv_unroll=unroll)
            sol, it, rr = sim.linear_solve(x, C, kappa, b, tol=1e-8)
            again, it2, _ = sim.linear_solve(x, C, kappa, b, tol=1e-8)
            assert it > 0 and it == it2 and np.array_equal(sol, again)
            assert rr <= 1e-8
            assert np.linalg.norm(H @ sol - b) <= 2e-8 * np.linalg.norm(b), (lanes, unroll)
    zero, it, _ = sim.linear_solve(x, C, kappa, np.zeros_like(b), tol=1e-8)
    assert it == 0 and not zero.any()
    sim.close()


@pytest.mark.parametrize("n,sheets", [(2, 1), (5, 1), (9, 3), (23, 1)])
def test_dense_direct_shapes(require_gpu, n, sheets):
    """one tile, a ragged last tile, several tiles of the dense factorisation and of the
    substitutions; the residual of a backward-stable solve is a small multiple of 2^-53"""
    sd, x, b = system(n, sheets)
    sim = Simulator(sd)
    C, kappa = sim.constraint_set(x), sim.scalars()["kappa"]
    H = sim.hessian(x, C, kappa)
    sim.set_linear_solver("direct")
    sol, _, rr = sim.linear_solve(x, C, kappa, b)
    assert np.linalg.norm(H @ sol - b) <= 1e-11 * np.linalg.norm(b), rr
    sim.close()

"""The 64-wide layers of the learned preconditioner on the FP32 matrix cores at sizes where
their tiles can go wrong: fewer rows than one tile of 16, ragged last tiles, fewer edges than
one row range of the weight gradient.

Bar: as in test_learned_gpu.py -- loss 1e-4, every parameter tensor's gradient 1e-3 relative
(FP32 against float64: sums of up to 10^5 terms of random sign lose about sqrt(n) 2^-24)."""
import numpy as np
import pytest

import learned_ref as R
import oracle as O
from cipc import Simulator, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 6, 17])
def test_loss_and_gradient_at_ragged_sizes(require_gpu, n):
    sd = scenes.cloth_on_sphere(sheets=1, n=n, y0=0.2008, sphere_level=0, seed=n)
    sim = Simulator(sd)
    orc = O.OracleScene(sd, threads=2)
    x = sd.X.ravel().copy()
    C = orc.constraint_set(x)
    kappa = orc.scalars()["kappa"]
    sim.precond_init(n)
    w = sim.precond_weights()
    L, _ = R.layout()
    rng = np.random.default_rng(n)
    for name in ("wo", "bo", "wd", "bd"):   # off zero, so that every layer gets a gradient
        o, m = L[name]
        w[o:o + m] = (rng.standard_normal(m) * 0.02).astype(np.float32)
    sim.precond_set_weights(w)
    loss, grad = sim.precond_loss_grad(x, C, kappa, n_probes=3, seed=5)
    a = orc.arrays()
    dbc = np.zeros(sd.nV, bool)
    dbc[sd.dbc_idx] = True
    loss_c, grad_c = R.loss_and_grad(orc.hessian(x, C, kappa, which=3), a["mass"], dbc, a["tri"], a["hinge"], w, 3, 5,
                                     R.contact_row_counts(sd.nV, C, dbc))
    assert abs(loss - loss_c) <= 1e-4 * (1 + abs(loss_c))
    for name, (o, m) in L.items():
        gc, gg = grad_c[o:o + m], grad[o:o + m].astype(np.float64)
        assert np.linalg.norm(gg - gc) <= 1e-3 * np.linalg.norm(gc) + 1e-9, name
    sim.close()

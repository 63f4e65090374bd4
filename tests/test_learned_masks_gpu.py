"""Rounding of the learned preconditioner's forward layers: every pre-activation is the chain
of fused multiply-adds b + x_0 w_0 + x_1 w_1 + ... in index order.  The gradient switches on
the sign of the pre-activations, so the order decides it where one stands within FP32
rounding of zero.  The weights of seeds 24, 88 and 195 hold such a unit: summed in another
order (groups of 16 inputs taken 0, 4, 8, 12, 1, 5, ...) one mask flips and the gradient moves
by 5.5e-3, 5.6e-4 and 1.0e-3 in 2-norm; seed 0 holds none.

Bar: 2e-6 in 2-norm against the float64 gradient with the masks of the FP32 chain.  With equal
masks only rounding is left: 9 layers forward and 9 back of chains of up to 192 products, for
terms of random sign sqrt(18 x 192) 2^-24 = 3.5e-6 if every chain kept its whole error; measured
1.3e-7 to 1.6e-7, and the smallest flip is 280 bars away."""
import numpy as np
import pytest
import torch

import learned_ref as R
import oracle as O
from cipc import Simulator, precond, scenes

pytestmark = pytest.mark.gpu


def chain(x, w, b):
    """FP32 b + sum_k x_k w_k, one rounding per product (exact in float64) and k"""
    acc = b.double().expand(len(x), -1)
    x, w = x.double(), w.double()
    for k in range(x.shape[1]):
        acc = torch.addcmul(acc, x[:, k:k + 1], w[k]).float().double()
    return acc.float()


def masks(node, ef, er, ec, weights):
    L, _ = R.layout()
    wq = torch.tensor(R.bf16(weights))
    out = {}

    def layer(name, x, w, b):
        z = chain(x, wq[L[w][0]:L[w][0] + L[w][1]].reshape(x.shape[1], -1), wq[L[b][0]:L[b][0] + L[b][1]])
        out[name] = z > 0
        return torch.where(out[name], z, torch.zeros(()))

    h = layer("h", torch.tensor(node.astype(np.float32)), "we", "be")
    e = layer("e", torch.tensor(ef.astype(np.float32)), "wx", "bx")
    for l in range(R.LAYERS):
        m = layer("m%d" % l, torch.cat([h[er], h[ec], e], 1), "wm%d" % l, "bm%d" % l)
        agg = np.zeros(h.shape, np.float32)
        np.add.at(agg, er, m.numpy())
        h, e = h + layer("u%d" % l, torch.cat([h, torch.tensor(agg)], 1), "wu%d" % l, "bu%d" % l), e + m
    return out


@pytest.mark.parametrize("seed", [0, 24, 88, 195])
def test_gradient_with_the_masks_of_the_sequential_chain(require_gpu, seed):
    n = 17
    sd = scenes.cloth_on_sphere(sheets=1, n=n, y0=0.21, sphere_level=0, seed=n)
    sim, orc = Simulator(sd), O.OracleScene(sd, threads=2)
    x, none = sd.X.ravel().copy(), np.zeros((0, 4), np.int32)
    w = precond.load()
    w = (w * (1 + 0.05 * np.random.default_rng(seed).standard_normal(w.shape))).astype(np.float32)
    sim.precond_set_weights(w)
    loss, grad = sim.precond_loss_grad(x, none, 1.0, n_probes=3, seed=5)
    sim.close()
    a = orc.arrays()
    dbc = np.zeros(sd.nV, bool)
    dbc[sd.dbc_idx] = True
    system = (orc.hessian(x, none, 1.0, which=3), a["mass"], dbc, a["tri"], a["hinge"])
    on = masks(*R.features(*system)[:4], w)
    loss_c, grad_c = R.loss_and_grad(*system, w, 3, 5, relu=lambda z, layer: z * on[layer])
    err = np.linalg.norm(grad - grad_c) / np.linalg.norm(grad_c)
    print("seed %d: loss %.2e gradient %.2e" % (seed, abs(loss - loss_c), err))
    assert abs(loss - loss_c) <= 1e-6 * (1 + abs(loss_c))
    assert err <= 2e-6

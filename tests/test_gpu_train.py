"""Training step of the closure's network at the edges of its kernels: batches
below, at and above 16 (samples of a block) and 128 (samples a weight's sum takes
at a time), rows taken through the epoch's order, batches without weight.

Bounds: the oracle rounds activations to FP16 as the kernel does, but from its own
FP64 values, so a few of them fall to the neighbouring FP16 number, 2^-11 of
themselves away: each is one of 128 terms, under 1e-3 of a gradient's norm and
(entering twice, with weights of 0.1) 1e-4 of the loss."""
import numpy as np
import pytest

import mlp as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


def _data(n):
    rng = np.random.default_rng(n)
    p = (0.1 * rng.standard_normal(M.NPAR)).astype(np.float32)
    return p, rng.standard_normal((n, M.IN)).astype(np.float32), rng.standard_normal((n, M.OUT)).astype(np.float32), rng.uniform(0.5, 2.0, n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 1000])
@pytest.mark.parametrize("weighted", [False, True])
def test_gradient_vs_oracle(vg, n, weighted):
    p, x, t, w = _data(n)
    w = w if weighted else None
    loss, g = vg.mlp_loss_grad(p, x, t, w)
    lref, gref = M.loss_grad(p, x, t, half=True, w=w)
    assert abs(loss - lref) <= 1e-4 * lref
    for a, b in [(M.OW1, M.OB1), (M.OB1, M.OW2), (M.OW2, M.OB2), (M.OB2, M.OW3), (M.OW3, M.OB3), (M.OB3, M.NPAR)]:
        assert np.linalg.norm(g[a:b] - gref[a:b]) < 1e-3 * np.linalg.norm(gref[a:b]), (a, b)


@pytest.mark.parametrize("n,batch", [(20, 1), (50, 7), (129, 128)])
def test_batches_without_weight_take_no_step(vg, n, batch):
    """One row has weight: an epoch is the one step that this row alone makes."""
    p, x, t, w = _data(n)
    w[:] = 0.0
    w[n // 2] = 1.5
    one = slice(n // 2, n // 2 + 1)
    par, loss = vg.mlp_train(p, x, t, 1, batch, 1e-3, seed=3, w=w)
    ref, lref = vg.mlp_train(p, x[one], t[one], 1, 1, 1e-3, seed=3, w=w[one])
    assert np.array_equal(par, ref) and loss[0] == pytest.approx(lref[0], rel=1e-6)

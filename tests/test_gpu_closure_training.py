"""The training kernels of the learned closure (k_mlp_grad, k_mlp_update) at the
edges of their 64-sample groups and of one group per compute unit, against
oracle/closure.py.

Tolerances: loss and gradient as in test_gpu_closure.py (BF16 operands with FP32
accumulation on both sides, other orders of summation).  What both calls compute
by the same operations in the same order is equal bit for bit.
"""
import numpy as np
import pytest

import closure as cl
from entropicthreadsafe_amd.tslb import Closure
from test_gpu_closure import _params, _samples

pytestmark = pytest.mark.gpu


def _drawn(seed, step, nb, ns):
    """The samples a training step draws: splitmix64 of (seed, step, j) mod ns."""
    with np.errstate(over="ignore"):
        x = np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(step) * np.uint64(0xD1B54A32D192ED03)
        x = x + np.arange(nb, dtype=np.uint64)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        x = x ^ (x >> np.uint64(31))
    return (x % np.uint64(ns)).astype(np.int32)


@pytest.mark.parametrize("nb", [1, 63, 64, 65, 16384, 16385, 33000])
def test_loss_and_gradient_at_group_edges(nb):
    th = _params(2)
    F, aux = _samples(40000, 4)
    with Closure(max_samples=40000) as m:
        m.set_params(th)
        m.set_samples(F.T, aux.T)
        loss, g = m.loss_grad(1e-3, idx=np.arange(nb, dtype=np.int32))
        m.clear_samples()
        m.set_samples(F[:nb].T, aux[:nb].T)  # no index list: all samples
        loss2, g2 = m.loss_grad(1e-3)
    assert loss2 == loss and np.array_equal(g2, g)
    lref, gref = cl.loss_and_grad(th, F[:nb], aux[:nb].astype(np.float64), 1e-3, emulate=True)
    print("loss", loss, lref, "grad rel", np.linalg.norm(g - gref) / np.linalg.norm(gref))
    assert abs(loss - lref) < 1e-3 * lref
    for a, b in ((0, 640), (640, 704), (704, 4800), (4800, 4864), (4864, 8960), (8960, 9024), (9024, 9472),
                 (9472, 9479)):
        assert np.linalg.norm(g[a:b] - gref[a:b]) < 5e-2 * np.linalg.norm(gref[a:b]) + 1e-30, (a, b)
    assert np.all(g[9479:] == 0)


@pytest.mark.parametrize("ns,nb", [(1, 70), (2, 64), (3, 1), (777, 5000), (40000, 20000)])
def test_training_step_draws_updates_and_repacks(ns, nb):
    th = _params(2)
    F, aux = _samples(ns, 4)
    with Closure(max_samples=ns) as m, Closure(max_samples=ns) as m2:
        for x in (m, m2):
            x.set_params(th)
            x.set_samples(F.T, aux.T)
        loss, g = m2.loss_grad(1e-3, idx=_drawn(7, 1, nb, ns))
        assert m.train(1, nb, 1e-3, 1e-3, seed=7) == loss  # the same samples, sums in the same order
        got = m.get_params()
        # first Adam step from zero moments: th - lr g / (|g| + eps), in FP32
        want = th - 1e-3 * (g / (np.abs(g) + 1e-8))
        assert np.abs(got - want).max() < 2e-7 + 4e-7 * np.abs(want).max()
        # the operands repacked in place are those of a full pack
        m2.set_params(got)
        assert np.array_equal(m.forward(), m2.forward())
        assert m.loss_grad(1e-3)[0] == m2.loss_grad(1e-3)[0]
        assert np.array_equal(m.loss_grad(1e-3)[1], m2.loss_grad(1e-3)[1])

"""What a training of the closure gives: the order of the sums over a batch and
Adam's arithmetic decide every bit of the trained weights.

golden/closure_training.npz holds the weights that the kernels trained which
added slices of 512 samples with atomics (`trained` below, run against that
build on an MI355X); with at most two slices a run of theirs repeated itself.
"""
import os

import numpy as np
import pytest

from entropicthreadsafe_amd.tslb import Closure
from test_gpu_closure import _params, _samples
from test_gpu_closure_training import _drawn

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "closure_training.npz")
BATCHES = (100, 600, 850, 1024)


def trained(nb, steps=60):
    F, aux = _samples(6000, 4)
    with Closure(max_samples=6000) as m:
        m.set_params(_params(2))
        m.set_samples(F.T, aux.T)
        m.train(steps, nb, 2e-3, 1e-3, seed=5)
        return m.get_params()


@pytest.mark.parametrize("nb", BATCHES)
def test_trained_weights_bit_for_bit(nb):
    want = np.load(GOLDEN)[f"theta_{nb}"]
    got = trained(nb)
    assert np.array_equal(got, want), np.abs(got - want).max()


@pytest.mark.parametrize("nb", [1024, 1536, 2048, 4096])
def test_gradient_is_the_sum_of_its_slices(nb):
    """Slices of 512, each a gradient of its own, added in order.  The weight of a
    sample is 1/nb, a power of two apart for the scaled batches below, so the
    scaling is exact."""
    F, aux = _samples(6000, 4)
    idx = np.random.default_rng(8).integers(0, 6000, nb).astype(np.int32)
    with Closure(max_samples=6000) as m:
        m.set_params(_params(2))
        m.set_samples(F.T, aux.T)
        # t_scale^2 nb is the same for the whole batch and its slices
        whole = m.loss_grad(2.0 ** -10, idx=idx)[1] if nb != 1536 else None
        parts = [m.loss_grad(2.0 ** -10, idx=idx[k:k + 512])[1] for k in range(0, nb, 512)]
        if nb == 1536:  # as 2048 with a slice repeated
            idx = np.concatenate([idx, idx[:512]])
            parts.append(parts[0])
            whole = m.loss_grad(2.0 ** -10, idx=idx)[1]
    want = np.zeros_like(whole)
    for g in parts:
        want = want + g * np.float32(512 / idx.size)
    assert np.array_equal(whole, want)


@pytest.mark.parametrize("nb", [300, 1500, 5000])
def test_adam_over_many_steps(nb):
    """Each of 25 steps against Adam in 64 bits on the gradient of the same samples.
    A step differs by the FP32 operations (a few 2^-24 relative) and by the
    power's last bit in 1 - 0.999^t, 2^-24 / (0.001 t) of it, half of that after
    the square root: 6e-5 / t allows two such bits."""
    ns, lr, b1, b2 = 6000, 2e-3, float(np.float32(0.9)), float(np.float32(0.999))
    F, aux = _samples(ns, 4)
    with Closure(max_samples=ns) as m, Closure(max_samples=ns) as m2:
        for x in (m, m2):
            x.set_samples(F.T, aux.T)
        m.set_params(_params(2))
        m1, v = np.zeros(9496), np.zeros(9496)
        for t in range(1, 26):
            th = m.get_params()
            m2.set_params(th)
            loss, g = m2.loss_grad(1e-3, idx=_drawn(7, t, nb, ns))
            g = g.astype(np.float64)
            m1 = b1 * m1 + (1 - b1) * g
            v = b2 * v + (1 - b2) * g * g
            want = lr * (m1 / (1 - b1 ** t)) / (np.sqrt(v / (1 - b2 ** t)) + 1e-8)
            assert m.train(1, nb, lr, 1e-3, seed=7) == loss
            got = th.astype(np.float64) - m.get_params()
            # FP32: the result is rounded to th's precision; m1 keeps 2^-24 of its
            # largest term through cancellations
            tol = (6e-5 / t + 2e-6) * lr + 2.0 ** -23 * np.abs(th) + 1e-12
            assert (np.abs(got - want) <= tol).all(), (t, (np.abs(got - want) / tol).max())

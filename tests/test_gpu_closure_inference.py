"""The closure fields of a lattice (k_features writing the first layer's operand,
k_mlp_infer<MlpPacked>) are bit for bit what the stored-sample path gives
(k_features writing FP32 inputs, k_mlp_infer<MlpPlain>, which
test_gpu_closure.py compares with the oracle): the same inputs, scaled and
rounded to BF16 by the same operations.  Samples taken with factor 1 are the
lattice's own nodes: rho u / rho of two FP32 values is exact in FP64.  Shapes
with partial tiles, a single tile and an odd number of them.
"""
import numpy as np
import pytest

import closure as cl
from entropicthreadsafe_amd.tslb import Closure, Lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 5), (16, 1, 1), (5, 3, 7), (33, 9, 5), (64, 4, 8), (70, 21, 11)])
@pytest.mark.parametrize("ncomp,storage,periodic", [(1, "fp32", (1, 1, 1)), (2, "fp32", (1, 0, 1)),
                                                    (2, "fp16", (1, 1, 0))])
def test_lattice_and_sample_paths_agree(shape, ncomp, storage, periodic):
    nx, ny, nz = shape
    rng = np.random.default_rng(7)
    th = cl.init_params(12, in_scale=np.array([5.0] * 6 + [3.0] * 3 + [1.0]),
                        out_scale=np.array([5e-3] + [2e-5] * 6))
    with Lattice(nx, ny, nz, ncomp=ncomp, tau=0.6, sigma=0.01 if ncomp == 2 else 0.0,
                 sharp_c=2.0 if ncomp == 2 else 0.0, periodic=periodic, storage=storage) as lat, Closure(nx * ny * nz) as m:
        m.set_params(th)
        for name, lo, hi in (("rho", 0.98, 1.02), ("u", -0.1, 0.1), ("v", -0.1, 0.1), ("w", -0.1, 0.1), ("phi", 0, 1)):
            lat.upload_field(name, rng.uniform(lo, hi, (nz, ny, nx)).astype(np.float32))
        lat.set_closure(m)
        got = lat.download_closure().reshape(7, -1)
        m.add_samples(lat, 1)
        want = m.forward()
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    assert np.array_equal(got, want)

"""The jet's inlet and outlet planes round every moment as the build with plain
moment fields did (golden/jet_states.txt: `state_hash` run against that build on
an MI355X).  They use the same operations as the fused pass, and which of two
products of a sum is fused shows in the last bit of 16-bit storage."""
import hashlib
import os

import numpy as np
import pytest

from entropicthreadsafe_amd.tslb import Lattice

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "jet_states.txt")
SHAPES = ((40, 36, 50), (128, 64, 16))
MODELS = {
    "1c": dict(ncomp=1, tau=0.6),
    "1c-forced": dict(ncomp=1, tau=0.6, force=(1e-5, 0.0, 0.0)),
    "1c-shifted": dict(ncomp=1, tau=0.6, force=(1e-5, 0.0, 0.0), force_mode=1),
    "2c": dict(ncomp=2, tau=0.7, sigma=0.01, sharp_c=0.9, lin_force=1e-4),
}
STORAGE = ("fp32", "fp16", "bf16", "fx16")


def state_hash(shape, model, storage, steps=6):
    nx, ny, nz = shape
    rng = np.random.default_rng(3)
    f = {k: (0.02 * rng.uniform(-1, 1, (nz, ny, nx))).astype(np.float32) for k in "uvw"}
    f["rho"] = (1 + 0.01 * rng.uniform(-1, 1, (nz, ny, nx))).astype(np.float32)
    f["phi"] = rng.uniform(0, 1, (nz, ny, nx)).astype(np.float32)
    fluid = np.ones((nz, ny, nx), np.int32)
    fluid[0] = fluid[-1] = fluid[:, 0] = fluid[:, -1] = fluid[:, :, 0] = fluid[:, :, -1] = 0
    with Lattice(nx, ny, nz, storage=storage, periodic=(0, 0, 0), **MODELS[model]) as lat:
        lat.set_isfluid(fluid)
        lat.set_jet_bc(True)
        for k, v in f.items():
            lat.upload_field(k, v)
        lat.init_equilibrium(True)
        lat.step(steps)
        return hashlib.sha256((lat.download() + np.float32(0)).tobytes()).hexdigest()  # -0 counts as 0


@pytest.mark.parametrize("storage", STORAGE)
@pytest.mark.parametrize("model", sorted(MODELS))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_state_bit_for_bit(shape, model, storage):
    want = dict(line.rsplit(" ", 1) for line in open(GOLDEN).read().splitlines())
    assert state_hash(shape, model, storage) == want["%dx%dx%d %s %s" % (*shape, model, storage)]

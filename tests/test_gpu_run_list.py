"""The list of interface runs and its two counters (phase-field model): whichever
pass lists (the fused one, or k_iface_list after a call that may change the
state), and whether a run goes to one block of k_curv_list or is split among
up to eight, a step gives the same bits."""
import numpy as np
import pytest

from entropicthreadsafe_amd.tslb import Lattice

pytestmark = pytest.mark.gpu
FIELDS = ("rho", "u", "v", "w", "phi")


def phase(nx, ny, nz, spheres, seed):
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    phi = np.zeros((nz, ny, nx), np.float32)
    for _ in range(spheres):
        c, r = rng.random(3) * (nx, ny, nz), rng.uniform(4, 8)
        phi[(x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2 < r * r] = 1
    return phi


def run(shape, spheres, storage, calls):
    with Lattice(*shape, ncomp=2, tau=0.6, sigma=0.02, sharp_c=2.1, storage=storage) as lat:
        lat.upload_field("phi", phase(*shape, spheres, 3))
        lat.init_equilibrium(True)
        for k in range(6):
            calls(lat, k)
            lat.step(1)
        return [lat.download_field(f) for f in FIELDS]


def nothing(lat, k):
    pass


def twice(lat, k):
    lat.normals()
    lat.normals()


def dense(lat, k):
    if k % 2:
        lat.download_normals()


def same_phi(lat, k):
    if k % 3 == 1:
        lat.upload_field("phi", lat.download_field("phi"))


# runs listed: a few (each split among eight blocks), some hundred, more than
# the resident blocks
@pytest.mark.parametrize("shape,spheres", [((24, 24, 24), 1), ((70, 45, 33), 6), ((128, 96, 128), 300)])
@pytest.mark.parametrize("storage", ["fp32", "fp16"])
def test_calls_between_steps_change_no_bits(shape, spheres, storage):
    want = run(shape, spheres, storage, nothing)
    for calls in (twice, dense, same_phi):
        got = run(shape, spheres, storage, calls)
        for f, a, b in zip(FIELDS, want, got):
            assert np.array_equal(a, b), (calls.__name__, f)

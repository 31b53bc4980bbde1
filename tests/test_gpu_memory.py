"""A lattice that just fits as plain fields is created, masked and stepped: where
the padding of the moment layout's rows does not fit, it is left out."""
import gc

import numpy as np
import pytest

from entropicthreadsafe_amd.tslb import Lattice, mem_info

pytestmark = pytest.mark.gpu

GB = 10**9


def fields(nz):
    rng = np.random.default_rng(2)
    return {k: (0.02 * rng.uniform(-1, 1, (nz, 96, 96))).astype(np.float32) for k in ("u", "v", "w")}


def run(nz, rep, masked):
    f = fields(nz)
    with Lattice(96, 96, nz * rep, ncomp=1, tau=0.7) as lat:
        if masked:
            isf = np.ones((nz, 96, 96), np.int32)
            isf[0, 40:50, 40:50] = 0
            lat.set_isfluid(np.tile(isf, (rep, 1, 1)))
        for k, v in f.items():
            lat.upload_field(k, np.tile(v, (rep, 1, 1)))
        lat.init_equilibrium(False)
        lat.step(3)
        return lat.download_field("u"), lat.device_bytes()


@pytest.mark.parametrize("masked", [False, True])
def test_lattice_that_fits_without_padding(masked):
    """96x96 planes: 88 B a node as plain fields, 115 B with whole tiles (8 more with
    a mask and its upload).  12960 of them, with room for 96 or 105 B a node."""
    torch = pytest.importorskip("torch")
    nz, rep = 30, 432
    ref, _ = run(nz, 1, masked)
    n = 96 * 96 * nz * rep
    hog = []
    try:
        while (left := mem_info()[0] - (105 if masked else 96) * n) > GB // 8:
            hog.append(torch.empty(min(left, 32 * GB), dtype=torch.uint8, device="cuda"))
        got, used = run(nz, rep, masked)
        assert used < 93 * n
        assert (got.reshape(rep, *ref.shape) == ref).all()
    finally:
        hog.clear()
        gc.collect()
        torch.cuda.empty_cache()

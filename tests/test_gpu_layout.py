"""The layouts of the state buffers (tiles in superpages, rows in sequence over
a plane, planes that share rows, planes beyond 32-bit offsets) hold the same
state and step it alike.  A periodic lattice that repeats a smaller one stays
its repetition bit for bit in FP32 storage (every node does the same
operations on the same values), so each shape is compared with a small lattice
in the first layout; uploads, downloads and checkpoints are compared in every
storage type."""
import numpy as np
import pytest

import pyoracle as po
from entropicthreadsafe_amd.tslb import FIELDS, Lattice
from parity import field_errors

pytestmark = pytest.mark.gpu

# base shape (nx, ny, nz), repetitions: what the repeated lattice covers
SHAPES = {
    "odd line of tiles": ((64, 8, 3), (13, 3, 2)),      # 39 tiles: the last line of 12 partly used
    "rows in sequence": ((9, 9, 6), (1, 1, 40)),        # 81 nodes a plane, 240 planes
    "two planes a row": ((7, 4, 5), (1, 1, 60)),
    "sixteen planes a row": ((2, 2, 3), (1, 1, 120)),
    "one column": ((1, 1, 5), (1, 1, 80)),
}
MODELS = {
    "1c": dict(ncomp=1, tau=0.6, force=(1e-5, 0.0, 0.0)),
    "2c": dict(ncomp=2, tau=0.7, sigma=0.01, sharp_c=0.9, lin_force=1e-4),
    "colour": dict(ncomp=3, tau=0.8, tau_b=0.6, sigma=0.01, beta=0.7),
}


def fields(shape, seed):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    f = {k: 0.02 * rng.uniform(-1, 1, (nz, ny, nx)) for k in ("u", "v", "w")}
    f["rho"] = 1.0 + 0.01 * rng.uniform(-1, 1, (nz, ny, nx))
    f["phi"] = rng.uniform(0, 1, (nz, ny, nx))
    return {k: v.astype(np.float32) for k, v in f.items()}


def tile(a, rep):
    return np.tile(a, rep[::-1])


def run(shape, f, kw, steps, isfluid=None):
    with Lattice(*shape, **kw) as lat:
        if isfluid is not None:
            lat.set_isfluid(isfluid)
        for k, v in f.items():
            lat.upload_field(k, v)
        lat.init_equilibrium(True)
        lat.step(steps)
        return lat.download(), lat.reduce()


@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("model", sorted(MODELS))
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_repeated_lattice_steps_alike(shape, model, solid):
    base, rep = SHAPES[shape]
    f = fields(base, 3)
    isf = None
    if solid:
        isf = np.ones(base[::-1], np.int32)
        isf[0, 0, 0] = 0
    big = tuple(n * r for n, r in zip(base, rep))
    ref, rsum = run(base, f, MODELS[model], 4, isf)
    got, gsum = run(big, {k: tile(v, rep) for k, v in f.items()}, MODELS[model], 4,
                    None if isf is None else tile(isf, rep))
    assert np.isfinite(ref).all()
    for q, name in enumerate(FIELDS):
        assert np.array_equal(got[q], tile(ref[q], rep)), name
    np.testing.assert_allclose(gsum, rsum * np.prod(rep), rtol=1e-9, atol=1e-9)


@pytest.mark.parametrize("shape", [(63, 9, 5), (65, 7, 4), (129, 17, 3), (64, 8, 2), (1, 8, 64)])
def test_tile_edges_match_oracle(shape):
    """The suite's bound against the FP64 oracle: 1e-5 of each group's scale."""
    f = fields(shape, 7)
    del f["phi"]
    kw = dict(ncomp=1, tau=0.8)
    got, _ = run(shape, f, kw, 5)
    o = po.Oracle(*shape, periodic=(1, 1, 1), dtype=np.float64, **kw)
    o.init(*[f[k].astype(np.float64) for k in ("rho", "u", "v", "w")], np.zeros(shape[::-1]), False)
    o.step(5)
    err = field_errors(got, o.moments())
    assert max(err.values()) <= 1e-5, err


@pytest.mark.parametrize("storage", ["fp32", "fp16", "bf16", "fx16"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_fields_come_back_in_node_order(shape, storage, tmp_path):
    base, rep = SHAPES[shape]
    big = tuple(n * r for n, r in zip(base, rep))
    # multiples of 2^-10 below 1/8 have 7 significant bits: exact in every storage type
    m = np.random.default_rng(5).integers(-127, 128, (11,) + big[::-1]).astype(np.float32) / np.float32(1024)
    m[0] += np.float32(1)
    path = str(tmp_path / "state")
    with Lattice(*big, ncomp=2, storage=storage) as lat:
        lat.upload(m)
        assert np.array_equal(lat.download(), m)
        plane = -m[4, 1]
        lat.upload_plane("pxx", 1, plane)
        m[4, 1] = plane
        lat.checkpoint_write(path, 1)
    with Lattice(*big, ncomp=2, storage=storage) as lat:
        lat.checkpoint_read(path)
        assert np.array_equal(lat.download(), m)


@pytest.mark.parametrize("model", ["1c", "2c"])
def test_plane_beyond_32_bit_offsets(model):
    """10240 x 10752 nodes in one plane: 4.7 GB of moments."""
    base, rep = (64, 48, 1), (160, 224, 1)
    f = fields(base, 9)
    ref, _ = run(base, f, MODELS[model], 2)
    big = tuple(n * r for n, r in zip(base, rep))
    with Lattice(*big, **MODELS[model]) as lat:
        for k, v in f.items():
            lat.upload_field(k, tile(v, rep))
        lat.init_equilibrium(True)
        lat.step(2)
        for q, name in enumerate(FIELDS):
            got = lat.download_field(name)
            assert (got.reshape(224, 48, 160, 64) == ref[q].reshape(1, 48, 1, 64)).all(), name

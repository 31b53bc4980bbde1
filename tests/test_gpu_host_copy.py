"""Large copies to and from callers' arrays go in chunks through pinned slots
on several threads (from 8 MB to the host, 256 MB from it).  Every value comes
back, at sizes around the limits and the chunk edges, and with several
lattices copying at once from their own threads (the slots serve one copy at a
time, the others take the plain path)."""
import threading

import numpy as np
import pytest

from entropicthreadsafe_amd.tslb import Lattice

pytestmark = pytest.mark.gpu


def check(shape, seed):
    nx, ny, nz = shape
    a = np.random.default_rng(seed).random((nz, ny, nx), dtype=np.float32)
    with Lattice(nx, ny, nz, ncomp=2) as lat:
        lat.upload_field("u", a)
        lat.upload_field("phi", -a)
        return np.array_equal(lat.download_field("u"), a) and np.array_equal(lat.download_field("phi"), -a)


# 4 bytes a node: sizes around 8 and 16 MiB, one node more than whole
# 64 KiB chunks, odd sizes, 268 MB (cut in both directions)
@pytest.mark.parametrize("shape", [(2048, 1023, 1), (2048, 1024, 1), (2047, 1026, 1), (2048, 2047, 1), (2048, 2048, 1), (2047, 2051, 1), (65537, 65, 1), (301, 130, 187),
                                   (521, 509, 257)])
def test_every_value_comes_back(shape):
    assert check(shape, 1)


def test_lattices_on_their_own_threads():
    ok = [None] * 4

    def work(i):
        ok[i] = all(check((240 + i, 160, 120), 10 * i + r) for r in range(3))

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert ok == [True] * 4

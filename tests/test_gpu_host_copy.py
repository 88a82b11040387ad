"""Downloads: short copies (direct) and long ones (a ring of 512 KiB slots,
from 32 MiB of doubles or 4 MiB of FP32 values that are widened) hand over the
same values, also with tails shorter than a slot and several threads at once."""
import threading

import numpy as np
import pytest

from tlbm_amd.gpu import Lattice

pytestmark = pytest.mark.gpu


# 75 full slots of 65536 doubles, ragged tails, a short copy
@pytest.mark.parametrize("q,dims", [(15, (64, 64, 80)), (15, (61, 59, 79)), (19, (61, 59, 67)), (27, (20, 18, 22))])
def test_populations_come_back(q, dims):
    n = int(np.prod(dims))
    f = np.random.default_rng(1).random((n, q))
    with Lattice(q, *dims, np.zeros(n, np.uint8), omega=1.0, storage="f64") as lat:
        lat.set_populations(f)
        assert np.array_equal(lat.populations(), f)


def _moments(dims, storage, fields):
    n = int(np.prod(dims))
    with Lattice(19, *dims, np.zeros(n, np.uint8), omega=1.2, storage=storage) as lat:
        lat.init_from_macros(*fields)
        lat.step(1)
        return list(lat.macros().values())


@pytest.mark.parametrize("tiles", [(4, 4, 6), (3, 5, 11)])
@pytest.mark.parametrize("storage", ["f32", "f16", "f64"])
def test_moments_of_a_periodic_box_repeat(storage, tiles):
    # the tiles of a periodic box hold the values of one of them, bit for bit
    # (FP16 rounds by node, so its tiles agree to the rounding of the storage)
    dims = (24, 17, 31)
    rng = np.random.default_rng(2)
    one = [0.02 * rng.standard_normal(dims[::-1]) for _ in range(3)] + [1 + 0.01 * rng.standard_normal(dims[::-1])]
    small = _moments(dims, storage, [v.ravel() for v in one])
    large = _moments([a * b for a, b in zip(dims, tiles)], storage, [np.tile(v, tiles[::-1]).ravel() for v in one])
    for a, b in zip(small, large):
        a = np.tile(np.asarray(a).reshape(dims[::-1]), tiles[::-1]).ravel()
        # FP16: 19 populations, each a relative 2^-11 of a deviation of at most 0.2 w
        assert np.abs(np.asarray(b).ravel() - a).max() <= (19 * 2.0 ** -11 * 0.2 if storage == "f16" else 0.0)


def test_threads_download_at_once():
    dims, q = (64, 64, 48), 27
    n = int(np.prod(dims))
    out = [None] * 3

    def run(k):
        f = np.random.default_rng(k).random((n, q))
        with Lattice(q, *dims, np.zeros(n, np.uint8), omega=1.0, storage="f64") as lat:
            lat.set_populations(f)
            out[k] = all(np.array_equal(lat.populations(), f) for _ in range(3))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert out == [True] * 3

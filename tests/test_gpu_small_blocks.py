"""FP64 steps on both sides of the lattice size where the workgroup changes
(2^20 nodes): a periodic box made of equal tiles holds the values of one tile,
bit for bit, since every node does the same operations."""
import numpy as np
import pytest

from tlbm_amd.gpu import Lattice

pytestmark = pytest.mark.gpu


def _run(q, dims, fields):
    n = int(np.prod(dims))
    with Lattice(q, *dims, np.zeros(n, np.uint8), omega=1.3, cs=0.1, storage="f64") as lat:
        lat.init_from_macros(*[f.ravel() for f in fields])
        for _ in range(3):
            lat.step(1)
        return lat.macros()


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("dims", [(32, 32, 255), (32, 32, 256), (35, 31, 257)])
def test_tiles_of_a_periodic_box_agree(q, dims):
    # two by two tiles: one x-y plane less than 2^20 nodes, 2^20, and more
    tiles = (2, 2, 1)
    rng = np.random.default_rng(q)
    one = [0.02 * rng.standard_normal(dims[::-1]) for _ in range(3)] + [1 + 0.01 * rng.standard_normal(dims[::-1])]
    small = _run(q, dims, one)
    large = _run(q, [a * b for a, b in zip(dims, tiles)], [np.tile(f, tiles[::-1]) for f in one])
    for k, a in small.items():
        assert np.array_equal(np.tile(a.reshape(dims[::-1]), tiles[::-1]).ravel(), large[k])

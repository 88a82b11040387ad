"""The two-step pass (tlbm_amd/csrc/lbm_pair.h) against single steps.

A call of several steps takes them two at a time where pair_plan says so, a
call of one step never does, so step(7) and seven calls step(1) from one
random state compare the two.  Lattices just large enough for the pass: last
tiles that overhang the lattice in x and y, z segments of unequal length, the
periodic wrap in x, y and z across tiles, walls, an obstacle across a tile's
edge, inlet (with and without a profile) and outlet, and both tile widths.

Both run the same node update on the same values, with every rounding written
out, so they agree bit for bit in every storage, with the network too."""
import numpy as np
import pytest

from tlbm_amd import closure, geometry
from tlbm_amd.gpu import Lattice
from tlbm_amd.workloads import DEFAULT_NETWORK

pytestmark = pytest.mark.gpu

CASES = [  # q, storage, dims, cs, network, inlet profile
    (19, "f32", (100, 78, 67), 0.0, False, True),
    (19, "f32", (28, 173, 117), 0.1, False, False),
    (19, "f64", (94, 71, 90), 0.1, False, False),
    (15, "f64", (64, 64, 97), 0.0, False, True),
    (15, "f32", (124, 50, 90), 0.1, False, False),
    (27, "f32", (60, 95, 101), 0.1, False, False),
    (19, "f32x", (124, 65, 64), 0.0, False, False),
    (27, "f32x", (124, 95, 90), 0.1, False, True),
    (19, "f32", (124, 118, 132), 0.0, True, True),
    (27, "f32", (128, 112, 107), 0.0, True, False),
]


@pytest.mark.parametrize("q,storage,dims,cs,network,profile", CASES,
                         ids=[f"q{c[0]}-{c[1]}-{'x'.join(map(str, c[2]))}{'-net' if c[4] else ''}" for c in CASES])
def test_two_step_pass_matches_single_steps(gpu_lib, q, storage, dims, cs, network, profile):
    nx, ny, nz = dims
    print(f"q={q} {storage} {dims} cs={cs} network={network}", flush=True)
    nd = geometry.channel(nx, ny, nz, walls=("left", "bottom") if q == 19 else (),
                          obstacles=[geometry.sphere(min(62, nx // 2), 12, nz // 3, 6),
                                     geometry.sphere(nx - 2, ny - 2, nz // 2, 4)])
    rng = np.random.default_rng(q + nx)
    out = []
    f0 = None
    for calls in ((7,), (1,) * 7):
        with Lattice(q, nx, ny, nz, nd, omega=1.0 / 0.56, u_lbm=0.04, cs=cs, storage=storage) as lat:
            if network:
                lat.set_closure(*closure.split_closure(closure.load_network(DEFAULT_NETWORK))[0])
            if profile:
                lat.set_inlet_profile(0.04 * (1.0 + 0.1 * np.sin(np.arange(nx * ny))))
            if f0 is None:
                f0 = lat.populations()
                f0 *= 1.0 + 0.02 * rng.standard_normal(f0.shape)
            lat.set_populations(f0)
            for n in calls:
                lat.step(n)
            red = lat.reduce()
            out.append((lat.populations(), lat.macros(), red["residual"], red["mass"]))
    (fa, ma, ra, sa), (fb, mb, rb, sb) = out
    assert np.array_equal(fa, fb)
    assert all(np.array_equal(ma[k], mb[k]) for k in ma)
    assert ra == rb and sa == sb

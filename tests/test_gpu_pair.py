"""The two-step pass (tlbm_amd/csrc/lbm_pair.h) against single steps.

A call of several steps takes them two at a time where pair_plan says so, a
call of one step never does, so a call of n steps and n calls of one from one
random state compare the two.  One lattice for every kernel that is built
(velocity set, storage, tile, with and without the network; test_pair_plan.py
holds which tile each takes and that none is left out), just large enough for
the pass: last tiles that overhang the lattice in x and y, z segments of
unequal length, the periodic wrap in x, y and z across tiles, walls, an
obstacle across a tile's edge, inlet (with and without a profile) and outlet.

Both run the same node update on the same values, with every rounding written
out, so they agree bit for bit in every storage, with the network too."""
import numpy as np
import pytest

from tlbm_amd import closure, geometry
from tlbm_amd.gpu import Lattice
from tlbm_amd.workloads import DEFAULT_NETWORK

pytestmark = pytest.mark.gpu

CASES = [  # q, storage, tile, dims, cs, network, inlet profile
    (15, "f64", 0, (188, 59, 27), 0.0, False, True),
    (15, "f32", 0, (188, 49, 67), 0.1, False, False),
    (15, "f32", 1, (92, 103, 27), 0.0, False, True),
    (15, "f32", 0, (252, 206, 91), 0.0, True, False),
    (15, "f32", 1, (252, 111, 127), 0.0, True, True),
    (15, "f32x", 0, (252, 47, 31), 0.0, False, False),
    (15, "f32x", 1, (220, 47, 35), 0.0, False, True),
    (19, "f64", 0, (92, 35, 111), 0.0, False, True),
    (19, "f64", 0, (62, 191, 70), 0.1, False, False),
    (19, "f32", 0, (124, 39, 61), 0.0, False, True),
    (19, "f32", 1, (120, 41, 63), 0.0, False, False),
    (19, "f32", 1, (248, 53, 47), 0.1, False, False),
    (19, "f32", 0, (316, 38, 168), 0.0, True, True),
    (19, "f32", 1, (220, 251, 35), 0.0, True, False),
    (19, "f32x", 0, (380, 34, 47), 0.0, False, False),
    (19, "f32x", 1, (220, 47, 53), 0.0, False, True),
    (19, "f32x", 1, (252, 159, 79), 0.1, False, False),
    (27, "f32", 0, (188, 54, 45), 0.0, False, False),
    (27, "f32", 0, (124, 142, 41), 0.1, False, True),
    (27, "f32", 1, (92, 123, 35), 0.0, False, True),
    (27, "f32", 0, (316, 135, 134), 0.0, True, False),
    (27, "f32", 1, (124, 143, 159), 0.0, True, True),
    (27, "f32x", 0, (124, 47, 125), 0.0, False, True),
]


def _compare(q, storage, dims, cs, network, profile, steps, **kw):
    nx, ny, nz = dims
    print(f"q={q} {storage} {dims} cs={cs} network={network}", flush=True)
    nd = geometry.channel(nx, ny, nz, walls=("left", "bottom") if q == 19 else (),
                          obstacles=[geometry.sphere(min(62, nx // 2), 12, nz // 3, 6),
                                     geometry.sphere(nx - 2, ny - 2, nz // 2, 4)])
    rng = np.random.default_rng(q + nx)
    out = []
    f0 = None
    for calls in ((steps,), (1,) * steps):
        with Lattice(q, nx, ny, nz, nd, omega=1.0 / 0.56, u_lbm=0.04, cs=cs, storage=storage, **kw) as lat:
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


@pytest.mark.parametrize("q,storage,tile,dims,cs,network,profile", CASES,
                         ids=[f"q{c[0]}-{c[1]}-tile{c[2]}-{'x'.join(map(str, c[3]))}{'-net' if c[5] else ''}"
                              for c in CASES])
def test_two_step_pass_matches_single_steps(gpu_lib, q, storage, tile, dims, cs, network, profile):
    _compare(q, storage, dims, cs, network, profile, 7)


@pytest.mark.parametrize("storage", ["f64", "f32", "f32x"])
@pytest.mark.parametrize("steps,kw", [(2, {}), (4, {}), (8, {}), (5, {"dynamics": 2}), (6, {"exact_weights": True})],
                         ids=["2", "4", "8", "no-relaxation", "exact-weights"])
def test_counts_and_options(gpu_lib, storage, steps, kw):
    dims = {"f64": (92, 35, 111), "f32": (120, 41, 63), "f32x": (220, 47, 53)}[storage]  # of CASES
    _compare(19, storage, dims, 0.0, False, True, steps, **kw)


@pytest.mark.parametrize("storage,nx,passes", [("f64", 92, {1: 1, 2: 2, 3: 2, 7: 4, 8: 5}), ("f16", 92, {1: 1, 7: 7}),
                                               ("f64", 93, {7: 7})])
def test_passes_are_counted(gpu_lib, storage, nx, passes):
    """Two steps a pass but for a call's last one or two; one where rows are
    no multiple of 16 bytes, in FP16 and while averages are on."""
    with Lattice(19, nx, 35, 111, np.zeros(nx * 35 * 111, np.uint8), omega=1.2, storage=storage) as lat:
        for steps, n in passes.items():
            before = lat.passes()
            lat.step(steps)
            assert lat.passes() - before == n
        lat.time_average(True)
        before = lat.passes()
        lat.step(7)
        assert lat.passes() - before == 7

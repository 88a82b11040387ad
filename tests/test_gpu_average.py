"""Time averages are the sums of the moments that each step's dump gives.

The step adds to the sums as it goes (with the network a second pass does);
`macros()` forms the same moments in a kernel of its own.  Both read the same
populations and sum them in the same order, so FP64 agrees bit for bit; with
the other storages a compiler may contract one product in one kernel and not
in the other, one rounding (2^-23 of the moment, FP32X 2^-52) per step."""
import numpy as np
import pytest

from tlbm_amd import closure, geometry
from tlbm_amd.gpu import Lattice
from tlbm_amd.workloads import DEFAULT_NETWORK

pytestmark = pytest.mark.gpu

STEPS = 5


@pytest.mark.parametrize("q", [15, 19, 27])
@pytest.mark.parametrize("storage,network", [("f64", False), ("f32", False), ("f16", False), ("f32x", False),
                                             ("f32", True), ("f16", True)])
@pytest.mark.parametrize("dims,lid,profile", [((33, 22, 35), False, True), ((64, 16, 32), True, False),
                                              ((5, 7, 9), False, False)])
def test_average_is_the_sum_of_the_moments(q, storage, network, dims, lid, profile):
    nx, ny, nz = dims
    nd = geometry.channel(nx, ny, nz, walls=("left", "bottom"),
                          obstacles=[geometry.sphere(nx // 2, ny // 2, nz // 2, 2)]).astype(np.uint8).ravel()
    if lid:
        nd[(nz // 3) * nx * ny + 3 * nx + 5:][:7] = 5
    rng = np.random.default_rng(q)
    start = [0.02 * rng.standard_normal(nd.size) for _ in range(3)] + [1 + 0.01 * rng.standard_normal(nd.size)]
    sums = []
    for averaged in (True, False):
        with Lattice(q, nx, ny, nz, nd, omega=1 / 0.56, u_lbm=0.04, cs=0.0 if network else 0.1,
                     storage=storage) as lat:
            if profile:
                lat.set_inlet_profile(0.04 * (1 + 0.1 * np.sin(np.arange(nx * ny))))
            if network:
                lat.set_closure(*closure.split_closure(closure.load_network(DEFAULT_NETWORK))[0])
            lat.init_from_macros(*start)
            if averaged:
                lat.time_average(True)
                lat.step(STEPS)
                got, n = lat.get_time_average()
                assert n == STEPS
                sums.append([got[k] for k in ("u", "v", "w", "rho")])
            else:
                total = [np.zeros(nd.size) for _ in range(4)]
                for _ in range(STEPS):
                    lat.step(1)
                    for a, b in zip(total, lat.macros().values()):
                        a += b
                sums.append(total)
    for a, b in zip(*sums):
        unit = {"f64": 0.0, "f32x": 2.0 ** -52}.get(storage, 2.0 ** -23)
        most = STEPS * unit * np.abs(b).max()
        assert np.abs(a - b).max() <= most

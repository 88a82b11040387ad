"""The bits of a run.

A flow near tau = 1/2 grows a last-bit difference of a kernel's arithmetic by
orders of magnitude in a few hundred steps, and FP16's stochastic rounding and
the network's bf16 units flip on one, so runs can be compared across versions
only if the arithmetic stays the same to the last bit.  Every rounding of the
kernels is written out (equilibrium_dev in tlbm_amd/csrc/lbm_kernels.h); these
hashes are those of the package's first version on MI355X, for every storage,
lattice, relaxation rule and node type, in single steps and in one call
(where the lattice takes it, in two steps per pass)."""
import hashlib

import numpy as np
import pytest

from tlbm_amd import closure, geometry
from tlbm_amd.gpu import Lattice
from tlbm_amd.workloads import DEFAULT_NETWORK

pytestmark = pytest.mark.gpu

# lattice, storage, dims, rule (bgk, Smagorinsky, network, exact weights, no
# relaxation), inlet profile: hashes of the populations after one step, its
# moments, the populations after nine more steps one by one and in one call
# (FP16: after eight more), and for bgk and smag the time average of the next
# three steps, the populations after them and, on even sizes, the box filter
EXPECTED = {
    "15_f16_33x29x31_bgk_0": "c5d87512 a47a4c92 8f9518ce 7a1bd08b d1207597",
    "15_f16_33x29x31_dyn2_0": "284a519f a47a4c92 b5ed6c86",
    "15_f16_33x29x31_exact_0": "3b71d405 a47a4c92 19524370",
    "15_f16_33x29x31_net_0": "70330c5b a47a4c92 fe554a13",
    "15_f16_33x29x31_smag_0": "470adad0 a47a4c92 ea8cfec2 fd167f50 32c8a269",
    "15_f16_40x24x36_bgk_1": "1bc9a042 3b148ff8 ee167c9a 2bd53916 fe3fdcae 3e24491d",
    "15_f16_40x24x36_smag_1": "74965f71 8782ae72 3706d928 d57f19ed 83df91c6 48671b7a",
    "15_f32_124x65x90_net_1": "b31d404e cd98f2c7 b3a64f39 b3a64f39",
    "15_f32_124x65x90_smag_1": "b52e2de1 cd98f2c7 4499bdae 4499bdae b7256ce3 dc460723",
    "15_f32_128x112x106_net_0": "0320b0ee 9a7da2d0 8178c482 8178c482",
    "15_f32_28x173x117_bgk_1": "f32a2815 3b9fa2cc 739af68e 739af68e fda39c11 33ff358a",
    "15_f32_33x29x31_bgk_0": "769e37e9 a41fc29d c63e5f21 c63e5f21 2c2b10cd 4630d21b",
    "15_f32_33x29x31_dyn2_0": "5812a63a a41fc29d bcdc7772 bcdc7772",
    "15_f32_33x29x31_exact_0": "2f03b98f a41fc29d f8ffffcd f8ffffcd",
    "15_f32_33x29x31_net_0": "cc18f358 a41fc29d 4523ed7a 4523ed7a",
    "15_f32_33x29x31_smag_0": "fd7aa361 a41fc29d 3b6c0bf4 3b6c0bf4 8d52717e cc91f4d8",
    "15_f32_40x24x36_bgk_1": "9af5877e 0b2a6f50 cd06fb8a cd06fb8a 7d152c71 ecda30bc 89f94197",
    "15_f32_40x24x36_smag_1": "3d917623 2fb4869d 02c6c431 02c6c431 eb27b538 b564f5d5 df97c7be",
    "15_f32x_124x65x90_smag_1": "140b2245 75f9b354 60207cd8 60207cd8 af41314c 5ca328e9",
    "15_f32x_28x173x117_bgk_1": "16b958b2 d398887f 2b63fe04 2b63fe04 64fec5fa 70f25dad",
    "15_f32x_33x29x31_bgk_0": "e89e8693 ffa5f217 448800e3 448800e3 941588ad 9b23c931",
    "15_f32x_33x29x31_dyn2_0": "84e272e7 ffa5f217 384746a3 384746a3",
    "15_f32x_33x29x31_exact_0": "586afe3b 9d248631 b6395e8a b6395e8a",
    "15_f32x_33x29x31_smag_0": "77063d26 ffa5f217 e2d35ceb e2d35ceb c4343e82 99d5c309",
    "15_f32x_40x24x36_bgk_1": "83fd94db 8334b1f8 72b41f2b 72b41f2b 24120cef 63ae6f52 c962680c",
    "15_f32x_40x24x36_smag_1": "4e07be64 24ae80d3 5e65c3cc 5e65c3cc a8a9cb15 39902369 c563fcdb",
    "15_f64_124x65x90_smag_1": "f6f23a3e bebea99a 1ec4641c 1ec4641c 55f4e180 1183df2f",
    "15_f64_33x29x31_bgk_0": "8f96d2af 9de0648b e332ea87 e332ea87 9b8b0d01 a1b6bb58",
    "15_f64_33x29x31_dyn2_0": "386da7b5 9de0648b 6feaa497 6feaa497",
    "15_f64_33x29x31_exact_0": "95d92db4 e51406e4 bfc7f8d7 bfc7f8d7",
    "15_f64_33x29x31_smag_0": "9d4abde5 9de0648b 1c2ed181 1c2ed181 03179e09 0cac72b4",
    "15_f64_40x24x36_bgk_1": "dab47659 26f1aa55 add36775 add36775 0681c483 4f00b57c fad57687",
    "15_f64_40x24x36_smag_1": "cf9d4f5b 5f625d16 1facb21d 1facb21d 3e13b601 9b7fe940 7fbd01c1",
    "19_f16_33x29x31_bgk_0": "3fef9291 0ba6636b 3876caaf 35f399a8 3e17935a",
    "19_f16_33x29x31_dyn2_0": "a5d343bf 0ba6636b 45bcacc2",
    "19_f16_33x29x31_exact_0": "889c277e 0ba6636b 75dd0923",
    "19_f16_33x29x31_net_0": "ab56be26 0ba6636b d1d14137",
    "19_f16_33x29x31_smag_0": "5b943aa0 0ba6636b f16662db 6dade7f1 e941a67d",
    "19_f16_40x24x36_bgk_1": "19cdec43 52f4969e 70237675 4d090250 1089f9f2 7bac334d",
    "19_f16_40x24x36_smag_1": "f866daa8 9f193849 44e7f4e3 6b6c43cd c6b7ef99 6b4ddd95",
    "19_f32_124x65x90_net_1": "460f7161 31d63814 3d0b167a 3d0b167a",
    "19_f32_124x65x90_smag_1": "943c24e0 31d63814 488f7c7b 488f7c7b fe9281f8 53bb3866",
    "19_f32_128x112x106_net_0": "1bc44329 359208fb 13b1757e 13b1757e",
    "19_f32_28x173x117_bgk_1": "c6d03147 6203dc29 7d9efb09 7d9efb09 3b3bac7c c17b3dde",
    "19_f32_33x29x31_bgk_0": "f14d713d 531ce709 221d6a93 221d6a93 de19f815 dd9979e7",
    "19_f32_33x29x31_dyn2_0": "75e22e7d 531ce709 4991cbe4 4991cbe4",
    "19_f32_33x29x31_exact_0": "78e204cc 531ce709 0d0e714e 0d0e714e",
    "19_f32_33x29x31_net_0": "30e943fd 531ce709 d3dbcc6a d3dbcc6a",
    "19_f32_33x29x31_smag_0": "a9161f6c 531ce709 aae0109c aae0109c b40ef777 38d81477",
    "19_f32_40x24x36_bgk_1": "0be184ef ff5d34ee af5bef34 af5bef34 78b74ce2 e3e018d4 1ebce8e6",
    "19_f32_40x24x36_smag_1": "7b194589 bf8b9787 92d932ad 92d932ad 3cb9f91c 31e39cb1 6fc24c27",
    "19_f32x_124x65x90_smag_1": "1b2c1a36 5104cc0d 2e58cc6d 2e58cc6d 7b347c71 bd090128",
    "19_f32x_28x173x117_bgk_1": "916125e0 ef91a5f6 05094809 05094809 682760d4 042264c7",
    "19_f32x_33x29x31_bgk_0": "b6c421f3 c259d24a 3a44b3e3 3a44b3e3 4b333046 75474cff",
    "19_f32x_33x29x31_dyn2_0": "0368b79a c259d24a 70083e5f 70083e5f",
    "19_f32x_33x29x31_exact_0": "00a86d17 4d2b25b5 19d57cc8 19d57cc8",
    "19_f32x_33x29x31_smag_0": "36934720 c259d24a 10dc6f8b 10dc6f8b b42b9561 57a52a4d",
    "19_f32x_40x24x36_bgk_1": "0876ff8b 6786857d f8186e20 f8186e20 0334e208 58009846 e6d3711f",
    "19_f32x_40x24x36_smag_1": "b18decaa 52ec7ac2 0cd7aae7 0cd7aae7 58ccbe23 eea1db7b 79a5366b",
    "19_f64_124x65x90_smag_1": "f3171e14 c571939b 01b29d58 01b29d58 81babdd6 0aee3e47",
    "19_f64_33x29x31_bgk_0": "60446867 2dedbcd7 952f9745 952f9745 d1281f04 da6e6d39",
    "19_f64_33x29x31_dyn2_0": "7b97feba 2dedbcd7 e8677cba e8677cba",
    "19_f64_33x29x31_exact_0": "f0eb4cc5 53c113b9 8b92c10a 8b92c10a",
    "19_f64_33x29x31_smag_0": "694c40c5 2dedbcd7 6698ea4b 6698ea4b 62ce7647 29ffc593",
    "19_f64_40x24x36_bgk_1": "c742ef32 7420520a b38336a9 b38336a9 7b1534fe 91d008ca 2e9cd08e",
    "19_f64_40x24x36_smag_1": "5c041779 cf7a0689 888eec0c 888eec0c c7bfa774 2547f148 53380e0b",
    "27_f16_33x29x31_bgk_0": "7c069e5c 21ddca54 2bafd2be a9359a87 1be202d7",
    "27_f16_33x29x31_dyn2_0": "42a04c8e 21ddca54 9c7256e3",
    "27_f16_33x29x31_exact_0": "7c069e5c 21ddca54 2bafd2be",
    "27_f16_33x29x31_net_0": "b338efd3 21ddca54 6a9d5106",
    "27_f16_33x29x31_smag_0": "cd09d7a4 21ddca54 76eec3f5 af449f7a 59e0262c",
    "27_f16_40x24x36_bgk_1": "259661ba 91192e19 ab5a4f29 7f14e8cc b89ea950 74da3545",
    "27_f16_40x24x36_smag_1": "4981e165 1a5d6f22 b5a1729f a9a5f48e a2434a20 3a68c1f1",
    "27_f32_124x65x90_net_1": "22bd0861 4da283e1 7e4efbea 7e4efbea",
    "27_f32_124x65x90_smag_1": "033d7919 4da283e1 8b12c8e2 8b12c8e2 7fc7a119 66d92925",
    "27_f32_128x112x106_net_0": "4bcdd8f1 0b32560e 79488f7c 79488f7c",
    "27_f32_28x173x117_bgk_1": "98d8de49 6e9d2ce2 1e2dd86d 1e2dd86d 5fcb9abd f6074c41",
    "27_f32_33x29x31_bgk_0": "11a5484b d29693fa 437ac618 437ac618 af8df329 c060ccda",
    "27_f32_33x29x31_dyn2_0": "6805f992 d29693fa 079d4aa7 079d4aa7",
    "27_f32_33x29x31_exact_0": "11a5484b d29693fa 437ac618 437ac618",
    "27_f32_33x29x31_net_0": "acb96aaf d29693fa d12125ec d12125ec",
    "27_f32_33x29x31_smag_0": "ec55facd d29693fa 3e976340 3e976340 85046a96 b75fcedd",
    "27_f32_40x24x36_bgk_1": "58ba04ae 4bb5274e 338abceb 338abceb 5896025b a76264f9 e763307d",
    "27_f32_40x24x36_smag_1": "b5431688 3d34a16b 0d2aac3b 0d2aac3b f0cf7b8b d84dae7e b9b27a4b",
    "27_f32x_124x65x90_smag_1": "4590a969 71dcce1f fe045f42 fe045f42 ab665f37 8e57606e",
    "27_f32x_28x173x117_bgk_1": "f6c25752 d37bb56e 28abf5dd 28abf5dd b352b54d ac7655cd",
    "27_f32x_33x29x31_bgk_0": "5f27e811 f7d8e5c5 c14c6626 c14c6626 51d3771d 77d3e6d0",
    "27_f32x_33x29x31_dyn2_0": "7c96dc16 f7d8e5c5 3eab4332 3eab4332",
    "27_f32x_33x29x31_exact_0": "5f27e811 f7d8e5c5 c14c6626 c14c6626",
    "27_f32x_33x29x31_smag_0": "991c155a f7d8e5c5 eb8a5cdf eb8a5cdf fb3e8f54 7af2743b",
    "27_f32x_40x24x36_bgk_1": "0aaf4a53 44e8118d 44c9a0ff 44c9a0ff a821af33 9178e571 38f67a9c",
    "27_f32x_40x24x36_smag_1": "d3b4b045 8a1715fd 0d7feafa 0d7feafa 48dacf07 2ba4fb1f b3c7ea4d",
    "27_f64_124x65x90_smag_1": "dc248d3b 8e8a8974 766451e1 766451e1 83f38fdd f89d6c7f",
    "27_f64_33x29x31_bgk_0": "b95161e8 4efb56c1 1dbdd264 1dbdd264 75357368 99e59b18",
    "27_f64_33x29x31_dyn2_0": "6ec4a9d6 4efb56c1 ef85e4c0 ef85e4c0",
    "27_f64_33x29x31_exact_0": "b95161e8 4efb56c1 1dbdd264 1dbdd264",
    "27_f64_33x29x31_smag_0": "326af788 4efb56c1 589886f3 589886f3 97469056 1a3fedc6",
    "27_f64_40x24x36_bgk_1": "fe513d62 744ccb67 71708f9a 71708f9a 273bf7e5 c73c450d 84ca384c",
    "27_f64_40x24x36_smag_1": "853ec5bc 2cc1bc91 d325147f d325147f d6605d68 2f265b96 6f5d7fb0",
}


def _hash(a):
    return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()[:8]


def _planes(fields):
    return _hash(np.concatenate([np.ravel(v) for v in fields.values()]))


@pytest.mark.parametrize("case", sorted(EXPECTED))
def test_bits_are_those_of_the_first_version(gpu_lib, case):
    q, storage, dims, rule, profile = case.split("_")
    nx, ny, nz = map(int, dims.split("x"))
    nd = np.array(geometry.channel(nx, ny, nz, walls=("left", "bottom"),
                                   obstacles=[geometry.sphere(min(62, nx // 2), 12, nz // 3, 6)]))
    if rule == "bgk" and profile == "1" and nx < 50:
        nd.reshape(nz, ny, nx)[10, :, 5:20] = 5
    print(case, flush=True)
    with Lattice(int(q), nx, ny, nz, nd, omega=1 / 0.53, u_lbm=0.04, cs=0.1 if rule == "smag" else 0.0,
                 storage=storage, exact_weights=rule == "exact", dynamics=2 if rule == "dyn2" else 1) as lat:
        if rule == "net":
            lat.set_closure(*closure.split_closure(closure.load_network(DEFAULT_NETWORK))[0])
        if profile == "1":
            lat.set_inlet_profile(0.04 * (1 + 0.1 * np.sin(np.arange(nx * ny))))
        f0 = lat.populations()
        f0 *= 1 + 0.02 * np.random.default_rng(1).standard_normal(f0.shape)
        lat.set_populations(f0)
        lat.step(1)
        got = [_hash(lat.populations())]
        got.append(_planes(lat.macros()))
        if storage == "f16":  # its rounding goes by the step count
            lat.step(8)
            got.append(_hash(lat.populations()))
        else:
            for calls in ((1,) * 9, (9,)):
                lat.set_populations(f0)
                for n in calls:
                    lat.step(n)
                got.append(_hash(lat.populations()))
        if rule in ("bgk", "smag"):
            lat.time_average(True)
            lat.step(3)
            got += [_planes(lat.get_time_average()[0]), _hash(lat.populations())]
            lat.time_average(False)
            if not (nx % 2 or ny % 2 or nz % 2):
                got.append(_planes(lat.box_filter()))
    assert " ".join(got) == EXPECTED[case]


# ... and the populations after 60 steps from a smooth flow, most of whose
# populations hardly leave their weights, so that the roundings of small
# corrections show (lattice, storage, rule)
SMOOTH = {
    "15_f32_bgk": "ba7da06e",
    "15_f32_smag": "39672cce",
    "15_f32_net": "17152900",
    "15_f16_bgk": "3d783361",
    "15_f16_net": "f1637843",
    "15_f32x_smag": "2ea28c9e",
    "19_f32_bgk": "b4c114dc",
    "19_f32_smag": "bd33ff07",
    "19_f32_net": "da115c60",
    "19_f16_bgk": "69be5cf6",
    "19_f16_net": "d40c161c",
    "19_f32x_smag": "7352baf6",
    "27_f32_bgk": "b6bd1b42",
    "27_f32_smag": "80208f65",
    "27_f32_net": "e63cf34d",
    "27_f16_bgk": "d39e3d4c",
    "27_f16_net": "cbd9264d",
    "27_f32x_smag": "5df634e0",
}


@pytest.mark.parametrize("case", sorted(SMOOTH))
def test_bits_of_a_smooth_flow(gpu_lib, case):
    q, storage, rule = case.split("_")
    nx, ny, nz = 128, 64, 64
    nd = np.array(geometry.channel(nx, ny, nz, walls=(), obstacles=[geometry.sphere(40, 30, 20, 6)]))
    x, y, z = (np.sin(2 * np.pi * np.arange(n) / n) for n in (nx, ny, nz))
    wave = 0.006 * (x[None, None, :] * y[None, :, None] * z[:, None, None]).ravel() * (nd != 1)
    with Lattice(int(q), nx, ny, nz, nd, omega=1 / 0.509, u_lbm=0.06, cs=0.1 if rule == "smag" else 0.0,
                 storage=storage) as lat:
        if rule == "net":
            lat.set_closure(*closure.split_closure(closure.load_network(DEFAULT_NETWORK))[0])
        lat.init_from_macros(wave, -wave, 0.06 * (nd != 1) + wave, 1.0 + 0.1 * wave)
        lat.step(60)
        assert _hash(lat.populations()) == SMOOTH[case]


@pytest.mark.parametrize("network", [False, True])
@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "f32x"])
@pytest.mark.parametrize("q", [15, 19, 27])
def test_solid_nodes_pass_on_any_value(gpu_lib, q, storage, network):
    """A solid node sends every population back the way it came and takes part
    in no arithmetic: a NaN or an infinity in one population of it shows up in
    one population, not in the others, with either relaxation rule."""
    if network and storage in ("f64", "f32x"):
        pytest.skip("the network runs in FP32 and FP16 storage")
    dims = (16, 12, 20)
    n = int(np.prod(dims))
    nd = np.zeros(dims[::-1], np.uint8)
    nd[9:12, 5:8, 7:10] = 1
    middle = 8 + dims[0] * (6 + dims[1] * 10)
    for bad in (np.nan, np.inf, -np.inf):
        with Lattice(q, *dims, nd.ravel(), omega=1.2, cs=0.1, storage=storage) as lat:
            if network:
                lat.set_closure(*closure.split_closure(closure.load_network(DEFAULT_NETWORK))[0])
            f = lat.populations().reshape(n, q)
            f[middle, 7] = bad
            lat.set_populations(f)
            lat.step(1)
            got = lat.populations().reshape(n, q)
        assert np.count_nonzero(~np.isfinite(got)) == 1

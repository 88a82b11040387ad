"""The two-step pass's division of a lattice (tlbm_amd/csrc/pair_plan.h), on the
host: every own column and every plane belongs to exactly one workgroup, the
tiles fit the kernel's, offsets stay in range, and the lattices of
test_gpu_pair.py take the pass in the tiles they name, each kernel's among
them."""
import os
import re
import subprocess
import tempfile

import test_gpu_pair

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r"""
#include <cstdio>
#include <cstdlib>
#include "pair_plan.h"
using namespace tlbm;
static int bad = 0;
// the tile, -1: single steps
static int check(uint32_t nx, uint32_t ny, uint32_t nz, int q, int storage, int rate) {
    PairPlan p{};
    const int size = storage == 0 ? 8 : 4;
    if (!pair_plan(nx, ny, nz, q, storage, PairRate(rate), 256, &p)) return -1;
    const PairShape s = pair_tile(q, storage, p.shape);
    bool ok = s.tx > 0 && nx % s.v == 0 && p.ty >= 1 && int(p.ty) <= s.ty;
    ok = ok && p.nseg >= 1 && p.nseg <= nz;
    // tiles cover x and y once: each starts inside the lattice, the last reaches its end
    ok = ok && uint64_t(p.ntx - 1) * s.tx < nx && uint64_t(p.ntx) * s.tx >= nx;
    ok = ok && uint64_t(p.nty - 1) * p.ty < ny && uint64_t(p.nty) * p.ty >= ny;
    // the block index decomposes by the two divisions
    const uint32_t tiles = p.ntx * p.nty, n = tiles * p.nseg;
    for (uint32_t b = 0; b < n; b += 1 + n / 997) {
        const uint32_t seg = udiv(b, p.div_tiles), t = b - seg * tiles, ty = udiv(t, p.div_ntx), tx = t - ty * p.ntx;
        ok = ok && seg < p.nseg && ty < p.nty && tx < p.ntx && tx + p.ntx * (ty + p.nty * seg) == b;
    }
    // planes: segments are consecutive and none is empty
    uint32_t at = 0;
    for (uint32_t k = 0; k < p.nseg; ++k) {
        const uint32_t z0 = uint64_t(k) * nz / p.nseg, z1 = uint64_t(k + 1) * nz / p.nseg;
        ok = ok && z0 == at && z1 > z0;
        at = z1;
    }
    ok = ok && at == nz;
    // largest lane offset from a plane's first chunk, 32 bits
    const uint64_t CH = 32768 / size, r = uint64_t(nx) * ny - 1 + CH - 1;
    ok = ok && (r + (r / CH) * (q - 1) * CH + (q - 1) * CH) * size < (uint64_t(1) << 32) && nx * uint64_t(ny) <= (1u << 25);
    if (!ok) { ++bad; std::printf("bad %u %u %u q%d storage %d\n", nx, ny, nz, q, storage); }
    return p.shape;
}
int main(int argc, char **argv) {
    for (int i = 1; i + 5 < argc; i += 6)
        std::printf("case %s %s %s %d\n", argv[i + 3], argv[i + 4], argv[i + 5], check(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), atoi(argv[i + 3]), atoi(argv[i + 4]), atoi(argv[i + 5])));
    const int qs[3] = {15, 19, 27};
    for (int q : qs)
        for (int storage = 0; storage < 4; ++storage)
            for (int k = 0; k < 4; ++k)
                if (pair_tile(q, storage, k).tx) std::printf("tile %d %d %d\n", q, storage, k);
    unsigned r = 12345;
    auto rnd = [&](unsigned n) { r = r * 1664525u + 1013904223u; return (r >> 8) % n; };
    int taken = 0, all = 0;
    for (int k = 0; k < 600; ++k) {
        const uint32_t nx = 1 + rnd(700), ny = 1 + rnd(500), nz = 1 + rnd(400);
        const int storage = int(rnd(3)) == 0 ? 0 : (rnd(2) ? 1 : 3);
        ++all;
        taken += check(rnd(2) ? nx : 4 * (1 + nx / 4), ny, nz, qs[rnd(3)], storage, rnd(storage == 1 ? 3 : 2)) >= 0;
    }
    check(4096, 8192, 60, 19, 1, 0);   // the largest plane
    if (check(4100, 8192, 60, 19, 1, 0) >= 0) ++bad;
    if (check(102, 64, 64, 19, 1, 0) >= 0) ++bad;  // rows of 408 bytes
    if (check(24, 24, 96, 15, 0, 0) >= 0) ++bad;   // too small to gain
    for (int q : qs)
        if (check(128, 128, 512, q, 2, 0) >= 0) ++bad;  // FP16 has no tile
    // measured slower than single steps in every division tried (us per two
    // steps in single steps and in the best): D3Q15 FP32 with Smagorinsky 26.8
    // and 27.7, 26.0 and 26.8, with the network 63.9 and 74.3; D3Q19 with
    // Smagorinsky FP32X 102 and 106, FP64 57.8 and 58.2; D3Q27 with the network
    // 144 and 157
    bad += check(128, 64, 64, 15, 1, 1) >= 0;
    bad += check(64, 64, 128, 15, 1, 1) >= 0;
    bad += check(160, 100, 90, 15, 1, 2) >= 0;
    bad += check(96, 84, 240, 19, 3, 1) >= 0;
    bad += check(128, 64, 64, 19, 0, 1) >= 0;
    bad += check(96, 84, 240, 27, 1, 2) >= 0;
    std::printf("taken %d of %d bad %d\n", taken, all, bad);
}
"""


def test_plans_divide_the_lattice():
    number = {"f64": 0, "f32": 1, "f32x": 3}
    args, want = [], []
    for q, storage, tile, dims, cs, network, _ in test_gpu_pair.CASES:
        rate = 2 if network else int(cs > 0)
        args += [*map(str, dims), str(q), str(number[storage]), str(rate)]
        want.append((q, number[storage], rate, tile))
    with tempfile.TemporaryDirectory() as tmp:
        src, exe = os.path.join(tmp, "probe.cpp"), os.path.join(tmp, "probe")
        with open(src, "w") as fh:
            fh.write(PROBE)
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "tlbm_amd", "csrc"), src, "-o", exe],
                       check=True)
        out = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout
    got = [tuple(map(int, m)) for m in re.findall(r"case (\d+) (\d+) (\d+) (-?\d+)", out)]
    assert got == want
    tiles = {tuple(map(int, m)) for m in re.findall(r"tile (\d+) (\d+) (\d+)", out)}
    kernels = {(*t, net) for t in tiles for net in (False, True) if not net or t[1] == 1}
    assert {(q, s, tile, rate == 2) for q, s, rate, tile in want} == kernels
    taken, total, bad = map(int, re.search(r"taken (\d+) of (\d+) bad (\d+)", out).groups())
    assert bad == 0 and taken > total // 4, out

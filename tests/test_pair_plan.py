"""The two-step pass's division of a lattice (tlbm_amd/csrc/pair_plan.h), on the
host: every own column and every plane belongs to exactly one workgroup, the
tiles fit the kernel's, offsets stay in range, and the lattices of
test_gpu_pair.py do take the pass."""
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
// the kernels' tiles (PairShapes)
static bool shape(int k, int q, int storage, PairShape &s) {
    if (storage == 0) { if (k || q == 27) return false; s = {32, 12, 2}; return true; }
    if (storage == 1) { if (k == 0) s = {64, q == 27 ? 8 : 13, 4}; else if (k == 1) s = {32, q == 27 ? 18 : 28, 4}; else return false; return true; }
    if (k == 0) s = {64, q == 27 ? 4 : 8, 4}; else if (k == 1) s = {32, q == 27 ? 12 : 20, 4}; else return false;
    return true;
}
static int bad = 0;
static bool check(uint32_t nx, uint32_t ny, uint32_t nz, int q, int storage, bool net) {
    PairPlan p{};
    const int size = storage == 0 ? 8 : 4;
    if (!pair_plan(nx, ny, nz, q, size, net, 256, [&](int k, PairShape &s) { return shape(k, q, storage, s); }, &p)) return false;
    PairShape s;
    bool ok = shape(p.shape, q, storage, s) && nx % s.v == 0 && p.ty >= 1 && int(p.ty) <= s.ty;
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
    return true;
}
int main(int argc, char **argv) {
    for (int i = 1; i + 5 < argc; i += 6)
        std::printf("case %d\n", check(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), atoi(argv[i + 3]), atoi(argv[i + 4]), atoi(argv[i + 5])));
    unsigned r = 12345;
    auto rnd = [&](unsigned n) { r = r * 1664525u + 1013904223u; return (r >> 8) % n; };
    int taken = 0, all = 0;
    for (int k = 0; k < 600; ++k) {
        const uint32_t nx = 1 + rnd(700), ny = 1 + rnd(500), nz = 1 + rnd(400);
        const int q[3] = {15, 19, 27};
        const int storage = int(rnd(3)) == 0 ? 0 : (rnd(2) ? 1 : 3);
        ++all;
        taken += check(rnd(2) ? nx : 4 * (1 + nx / 4), ny, nz, q[rnd(3)], storage, storage == 1 && rnd(2));
    }
    check(4096, 8192, 60, 19, 1, false);   // the largest plane
    if (check(4100, 8192, 60, 19, 1, false)) ++bad;
    if (check(102, 64, 64, 19, 1, false)) ++bad;  // rows of 408 bytes
    if (check(24, 24, 96, 15, 0, false)) ++bad;   // too small to gain
    std::printf("taken %d of %d bad %d\n", taken, all, bad);
}
"""


def test_plans_divide_the_lattice():
    args = []
    for q, storage, dims, _, network, _ in test_gpu_pair.CASES:
        args += [*map(str, dims), str(q), {"f64": "0", "f32": "1", "f32x": "3"}[storage], str(int(network))]
    with tempfile.TemporaryDirectory() as tmp:
        src, exe = os.path.join(tmp, "probe.cpp"), os.path.join(tmp, "probe")
        with open(src, "w") as fh:
            fh.write(PROBE)
        subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "tlbm_amd", "csrc"), src, "-o", exe],
                       check=True)
        out = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout
    assert out.count("case 1") == len(test_gpu_pair.CASES), out
    taken, total, bad = map(int, re.search(r"taken (\d+) of (\d+) bad (\d+)", out).groups())
    assert bad == 0 and taken > total // 4, out

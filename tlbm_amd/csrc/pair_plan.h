// pair_plan.h -- how the two-step pass (lbm_pair.h) divides a lattice, and
// whether it is faster there than two single steps.  Plain C++ (host tests).
#pragma once

#include <stdint.h>

#include "udiv.h"

namespace tlbm {

// A tile the pass is built for: at most tx x ty columns, rows of a multiple
// of v nodes (16 bytes).
struct PairShape {
    int tx, ty, v;
};

// The pass's division of the lattice.
struct PairPlan {
    int shape;                // the tile
    uint32_t ty;              // rows of a tile, at most the shape's
    uint32_t ntx, nty, nseg;  // tiles in x and y, segments in z
    UDiv div_ntx, div_tiles;
};

// Estimated time of one pass (two steps) in us: rounds of workgroups, one per
// CU, times the planes each marches through (its segment and one more at
// either end), times a plane's time.  That is at least the work between the
// barriers (2.4 us and 0.105 us per row of 32 D3Q19 columns; FP64 2.0 and
// 0.35), and at least 1.2 us more than the loads and stores, rims included, of
// the workgroups side by side take at 6.3 TB/s (9 where both state buffers fit
// the 256 MB cache).  Measured against it (us per pass): D3Q19 FP32
// 128x128x512 in 64x13 tiles and 12 segments 285 (estimate 302), 32x26 and 12
// 315 (308), 32x19 and 9 325 (330); 96x84x240 64x12 and 18 81 (85), 32x12 and
// 10 109 (95); 128x64x64 64x13 and 25 25 (27), 32x8 and 8 35 (32); FP64
// 128x128x512 32x12 and 11 639 (635), 32x10 and 4 711 (716); D3Q27 FP32 192^3
// 64x8 and 7 386 (397).
// With the learned closure a plane takes 1.1 to 1.7 us more (128x128x512 64x13
// and 12: 335 against 284 us per pass).
inline double pair_cost(uint32_t nx, uint32_t ny, uint32_t nz, int q, int size, bool network, uint32_t cus,
                        const PairShape &s, const PairPlan &p) {
    const double groups = double(p.ntx) * p.nty * p.nseg;
    const double rounds = double((uint64_t(p.ntx) * p.nty * p.nseg + cus - 1) / cus);
    const double planes = double((nz + p.nseg - 1) / p.nseg) + 2.0;
    const double wide = double(nx) / p.ntx, column = double(q) * size;
    const double bytes = column * ((wide + 2 * s.v) * (p.ty + 2) + wide * p.ty);
    const double state = 2.0 * double(nx) * ny * nz * column;
    const double rate = state < 200e6 ? 9.0e6 : 6.3e6;  // bytes per us
    const double rows = double(p.ty) * s.tx / 32.0;
    const double work = (size == 8 ? 2.0 + 0.35 * rows : 2.4 + 0.105 * rows) * q / 19.0;
    const double move = 1.2 + bytes * (groups / rounds) / rate;
    return rounds * planes * ((work > move ? work : move) + (network ? 1.4 : 0.0)) + 0.5;
}

// Chooses the division with the least estimated time; false if the pass
// cannot run (rows that are no multiple of 16 bytes, planes too large for its offsets)
// or two single steps (6 TB/s and 2.5 us each) are estimated no slower.
template <class F>  // bool shape(int k, PairShape &)
inline bool pair_plan(uint32_t nx, uint32_t ny, uint32_t nz, int q, int size, bool network, uint32_t cus, F shape,
                      PairPlan *out) {
    const double column = double(q) * size;
    // a node's index in its plane has 25 bits; lane offsets from a plane's
    // first chunk reach the plane and a 32 KiB run per direction either side
    if (uint64_t(nx) * ny > (1u << 25) || (double(nx) * ny + 3.0 * 32768.0 / size) * column >= 4294967296.0)
        return false;
    // below 30 MB of state a pass has gained nowhere (48x48x64 FP32 D3Q19, 22
    // MB: 13.7 against 13.4 us per two steps; 64^3, 40 MB: the same)
    if (2.0 * double(nx) * ny * nz * column < 30e6) return false;
    const double single = 2.5 + 2.0 * double(nx) * ny * nz * column / 6.0e6;
    double best = 0.97 * 2.0 * single;
    bool found = false;
    PairShape s;
    for (int k = 0; shape(k, s); ++k) {
        if (nx % uint32_t(s.v)) continue;
        PairPlan p{};
        p.shape = k;
        p.ntx = (nx + uint32_t(s.tx) - 1) / uint32_t(s.tx);
        const uint32_t least = (ny + uint32_t(s.ty) - 1) / uint32_t(s.ty);
        for (uint32_t n = least; n <= ny && n <= 2 * least + 2; ++n) {
            p.ty = (ny + n - 1) / n;
            p.nty = (ny + p.ty - 1) / p.ty;
            const uint64_t tiles = uint64_t(p.ntx) * p.nty;
            if (tiles >= (1u << 24)) continue;
            for (p.nseg = 1; p.nseg <= nz && (p.nseg == 1 || tiles * p.nseg <= 6 * uint64_t(cus)); ++p.nseg) {
                const double c = pair_cost(nx, ny, nz, q, size, network, cus, s, p);
                if (c < best) {
                    best = c;
                    *out = p;
                    found = true;
                }
            }
        }
    }
    if (found) {
        out->div_ntx = udiv_magic(out->ntx);
        out->div_tiles = udiv_magic(out->ntx * out->nty);
    }
    return found;
}

}  // namespace tlbm

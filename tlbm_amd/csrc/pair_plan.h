// pair_plan.h -- how the two-step pass (lbm_pair.h) divides a lattice, and
// whether it is faster there than two single steps.  Plain C++ (host tests).
#pragma once

#include <stdint.h>

#include "udiv.h"

namespace tlbm {

// A tile the pass is built for: at most tx x ty columns, rows of a multiple
// of v nodes (16 bytes).  tx = 0: none.
struct PairShape {
    int tx, ty, v;
};

// The k-th tile (k = 0, 1) of a lattice of q directions in a storage
// (TLBM_STORAGE_*); the second is for lattices whose width the first fits
// badly.  Each is as large as LDS (160 KiB) and the registers of one workgroup
// per CU allow.  FP16 and D3Q27 FP64 have none: FP16's pair of steps takes
// as long as two steps (D3Q19 128x128x512: 103 against 102 us per step), D3Q27
// FP64 did not fit 256 registers when it was tried (806 against 502 us).
constexpr PairShape pair_tile(int q, int storage, int k) {
    if (k < 0 || k > 1) return {};
    if (storage == 0 && q != 27 && k == 0) return {32, 12, 2};
    if (storage == 1) return k == 0 ? PairShape{64, q == 27 ? 8 : 13, 4} : PairShape{32, q == 27 ? 18 : 28, 4};
    if (storage == 3 && q == 27) return k == 0 ? PairShape{32, 12, 4} : PairShape{};
    if (storage == 3) return k == 0 ? PairShape{64, 8, 4} : PairShape{32, 20, 4};
    return {};
}

// What sets a node's relaxation rate in a step.
enum PairRate { kRateBgk, kRateSmagorinsky, kRateNetwork };

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
// barriers, so much per direction and so much for the rate, each with a share
// per row of 32 columns, and at least 1.2 us more than the loads and stores,
// rims included, of the workgroups side by side take at 6.3 TB/s (9 where both
// state buffers fit the 256 MB cache).  The work's coefficients are fitted to
// passes over 7 lattices of 2.6e5 to 8.4e6 nodes in up to 12 divisions each,
// every velocity set, storage and rate: 6 % from the measured time in the
// mean, 30 % at most.  With them the plans of those lattices are 0.9 % slower
// in the mean than the best of the divisions and of single steps, 10 % at most,
// and 2 % at most slower than single steps.  us per pass, measured (estimated):
// D3Q19 FP32 128x128x512 in 64x13 tiles and 12 segments 297 (304), 96x84x240
// 32x28 and 28 83 (84), 128x64x64 64x13 and 25 28 (27); with Smagorinsky 314
// (304), 86 (84), 31 (34); with the network 367 (387), 98 (100), 38 (43); FP64
// 128x128x512 32x12 and 11 640 (643); D3Q27 FP32 256x128x128 64x8 and 4 228
// (225), with Smagorinsky 253 (233).
inline double pair_cost(uint32_t nx, uint32_t ny, uint32_t nz, int q, int storage, PairRate rate, uint32_t cus,
                        const PairShape &s, const PairPlan &p) {
    const int size = storage == 0 ? 8 : 4;
    const double groups = double(p.ntx) * p.nty * p.nseg;
    const double rounds = double((uint64_t(p.ntx) * p.nty * p.nseg + cus - 1) / cus);
    const double planes = double((nz + p.nseg - 1) / p.nseg) + 2.0;
    const double wide = double(nx) / p.ntx, column = double(q) * size;
    const double bytes = column * ((wide + 2 * s.v) * (p.ty + 2) + wide * p.ty);
    const double state = 2.0 * double(nx) * ny * nz * column;
    const double hbm = state < 200e6 ? 9.0e6 : 6.3e6;  // bytes per us
    const double rows = double(p.ty) * s.tx / 32.0;
    double work = (storage == 0 ? 2.0 + 0.38 * rows : storage == 1 ? 2.4 + 0.115 * rows : 1.0 + 0.24 * rows) * q / 19.0;
    if (rate == kRateSmagorinsky)
        work += storage == 0 ? 0.1 * rows : storage == 1 ? 0.05 * rows : 0.75 + 0.03 * rows;
    else if (rate == kRateNetwork)
        work += (0.6 + 0.1 * rows) * (q == 27 ? 1.15 : 1.0);
    const double move = 1.2 + bytes * (groups / rounds) / hbm;
    return rounds * planes * (work > move ? work : move) + 0.5;
}

// Chooses the division with the least estimated time; false if the pass
// cannot run (rows that are no multiple of 16 bytes, planes too large for its offsets)
// or two single steps (6 TB/s and 2.5 us each) are estimated no slower.
inline bool pair_plan(uint32_t nx, uint32_t ny, uint32_t nz, int q, int storage, PairRate rate, uint32_t cus,
                      PairPlan *out) {
    const int size = storage == 0 ? 8 : 4;
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
    for (int k = 0; k < 2; ++k) {
        const PairShape s = pair_tile(q, storage, k);
        if (!s.tx || nx % uint32_t(s.v)) continue;
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
                const double c = pair_cost(nx, ny, nz, q, storage, rate, cus, s, p);
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

// lbm_pair.h -- two time steps in one pass over the lattice.
//
// A step of k_lbm reads and writes every population once and runs near the
// HBM's copy rate, so only moving fewer bytes makes it faster.  k_lbm_pair
// takes the lattice from B_n to B_{n+2} with one read and one write: a
// workgroup owns a tile of TX x ty columns (x, y) with a rim of one column
// around it, one thread per column, and marches along z.  At plane p it
//   1. gathers and collides step n+1 at plane p in every column, rim included,
//   2. hands the populations that leave a column sideways to the neighbour
//      columns through LDS (a population that keeps its column stays in its
//      register),
//   3. collides step n+2 at plane p-1 in the tile's own columns, whose
//      arrivals from planes p-2, p-1 and p are complete now, and writes it.
// Populations with e_z = 0 wait one plane in registers, those with e_z = +1
// two.
//
// The populations of plane p + 1 come to LDS by direct loads, 16 bytes a
// lane, that go out as soon as plane p's are in registers and land while
// plane p is worked on.  Gathered into registers instead (each lane its own
// 19 sources, shifted by +-1 in x), a cache line is asked for by several
// wavefronts while it is still on its way, which holds up the L1.
//
// Each node runs the very update of k_lbm (NET: of k_lbm_closure) in both
// steps in the same roundings, so the results are those of two
// single steps bit for bit.
//
// us per step, single steps -> this: D3Q19 128x128x512 FP32 201.5 -> 148.8
// (Smagorinsky 157.4, network 184.8), FP64 401 -> 317.5, FP32X 201 -> 159.8;
// D3Q15 FP32 163.2 -> 122.3; D3Q27 FP32 192^3 248 -> 220.  What bounds it is
// the one workgroup per CU, in lock step between three barriers a plane; LDS
// and registers leave no room for a second to fill its waits.  No unit is
// full: VALU issue is 47 (FP64) to 75 % busy (D3Q27 with Smagorinsky; 84 with
// the network), LDS 8 to 11 % (26), and HBM moves 4.0 to 4.4 TB/s.
#pragma once

#include <type_traits>

#include "lbm_kernels.h"
#include "pair_plan.h"

namespace tlbm {

// Populations that leave their column (they go through LDS), numbered.
template <class L>
constexpr bool pair_moves(int s) { return L::ex[s] != 0 || L::ey[s] != 0; }
template <class L>
constexpr int pair_slot(int s) {
    int n = 0;
    for (int k = 0; k < s; ++k) n += pair_moves<L>(k) ? 1 : 0;
    return n;
}

// The K-th tile's kernel: TX x TY own columns, the threads and the LDS they take.
template <class L, int ST, int K>
struct PairTile {
    static constexpr PairShape kShape = pair_tile(L::Q, ST, K);
    static constexpr int TX = kShape.tx, TY = kShape.ty;
    static constexpr int W = TX + 2, H = TY + 2;      // with the rim
    static constexpr int kOwn = (TX * TY + 63) / 64 * 64;  // the own columns' threads, whole wavefronts
    static constexpr int kRim = 2 * W + 2 * TY;
    static constexpr int BS = (kOwn + kRim + 63) / 64 * 64;
    static constexpr int kSize = int(sizeof(typename StorageT<ST>::st));
    static constexpr int V = kShape.v;                // values of a 16-byte load
    static_assert(V * kSize == 16, "whole 16-byte loads");
    static constexpr int SW = TX + 2 * V;             // staged row: x0 - V .. x0 + TX + V - 1
    static constexpr int kStage = L::Q * H * SW;      // staged values
    static constexpr int NS = pair_slot<L>(L::Q);
    static constexpr size_t kLds = size_t(kStage + NS * W * H) * kSize;
    static_assert(kLds <= 160 * 1024, "LDS of a CU");
};

// s_waitcnt vmcnt(0), other counters free: every load and store sent has landed.
__device__ inline void wait_vmcnt() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// The workgroup's barrier for LDS traffic: this wavefront's LDS accesses are
// done before it (global loads and stores stay in flight).
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Direct load of 16 bytes per lane: lane l's go to LDS byte dst + 16 l (dst
// uniform in the wavefront).
__device__ inline void load_lds(const void *src, void *dst) {
    using gptr = const __attribute__((address_space(1))) void *;
    using lptr = __attribute__((address_space(3))) void *;
    __builtin_amdgcn_global_load_lds((gptr)src, (lptr)dst, 16, 0, 0);
}

template <class L, int ST, class TL, bool NET>
__global__ void __launch_bounds__(TL::BS)
k_lbm_pair(const typename StorageT<ST>::st *__restrict__ fin, typename StorageT<ST>::st *__restrict__ fout,
           const uint8_t *__restrict__ nd_type, PairPlan pl, StepArgs a) {
    using S = StorageT<ST>;
    using T = typename S::T;
    using st = typename S::st;
    static_assert(ST != ST_F16, "no stochastic rounding here");
    constexpr int Q = L::Q;
    constexpr uint32_t kSize = sizeof(st);
    constexpr int CB = S::kCB;
    constexpr uint32_t CH = 1u << CB;
    constexpr int W = TL::W, H = TL::H, SW = TL::SW, V = TL::V, BS = TL::BS;
    __shared__ alignas(16) st lds[TL::kStage + TL::NS * W * H];
    st *const stage = lds, *const swap = lds + TL::kStage;
    __shared__ std::conditional_t<NET, MlpPacked, int> smlp;
    if constexpr (NET) {
        static_assert(sizeof(MlpPacked) <= 16u * BS, "one 16-byte load per lane");
        stage_network(a.mlp, &smlp);
    }

    const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t seg = udiv(b, pl.div_tiles);
    const uint32_t tile = b - seg * pl.ntx * pl.nty;
    const uint32_t tyi = udiv(tile, pl.div_ntx), txi = tile - tyi * pl.ntx;
    const uint32_t x0 = txi * TL::TX, y0 = tyi * pl.ty;
    const int z0 = int(uint64_t(seg) * a.nz / pl.nseg), z1 = int(uint64_t(seg + 1) * a.nz / pl.nseg);
    const uint32_t tid = threadIdx.x;

    // This thread's column (i, j) of the W x H grid, the node (x0 - 1 + i,
    // y0 - 1 + j) modulo the lattice: own columns by rows, then the rim.
    uint32_t i, j;
    if (tid < uint32_t(TL::kOwn)) {
        i = tid % TL::TX + 1;
        j = tid / TL::TX + 1;
    } else {
        const uint32_t r = tid - TL::kOwn;
        if (r < uint32_t(2 * W)) {
            i = r < uint32_t(W) ? r : r - W;
            j = r < uint32_t(W) ? 0 : pl.ty + 1;
        } else {
            const uint32_t k = r - 2 * W;
            i = (k & 1u) ? W - 1 : 0;
            j = (k >> 1) + 1;
        }
    }
    const bool live = j <= pl.ty + 1;  // a column of the tile or its rim
    if (!live) j = 0;
    const bool own = live && tid < uint32_t(TL::TX * TL::TY) && j <= pl.ty && x0 + i <= a.nx && y0 + j <= a.ny;
    const bool wave_own = __any(own);
    const uint32_t x = (x0 + i + a.nx - 1) % a.nx, y = (y0 + j + a.ny - 1) % a.ny;
    const uint32_t gxy = y * a.nx + x;
    const st *const sp = stage + j * SW + i + V - 1;          // own column's staged values
    st *const wp = swap + j * W + i;

    // What this thread loads: unit k of the staged box is V values (16 bytes)
    // at LDS byte 16 k.  The staged row j of direction s holds row
    // y0 - 1 + j - e_y.  nx is a multiple of V, so a unit neither wraps nor
    // straddles a chunk.
    constexpr int kUnits = TL::kStage / V;
    constexpr int kRowUnits = SW / V;
    constexpr int NI = (kUnits + BS - 1) / BS;
    // node in its plane (bits 0-24), direction (25-29), e_z + 1 (30-31; 3: no load)
    uint32_t unit[NI];
#pragma unroll
    for (int n = 0; n < NI; ++n) {
        const uint32_t k = uint32_t(n) * BS + tid;
        const uint32_t s = k / (H * kRowUnits), q = k - s * (H * kRowUnits);
        const uint32_t row = q / kRowUnits, u = q - row * kRowUnits;
        int ey = 0, ez = 0;
#pragma unroll
        for (int d = 0; d < Q; ++d)
            if (uint32_t(d) == s) { ey = L::ey[d]; ez = L::ez[d]; }
        const uint32_t xv = u * V;  // value within the row, from x0 - V
        // rows and values past the last column that is needed are left out
        const bool need = k < uint32_t(kUnits) && row <= pl.ty + 1 && x0 + xv <= a.nx + 1 + V &&
                          y0 + row <= a.ny + 1;
        const uint32_t xx = (x0 + xv + V * a.nx - V) % a.nx;
        const uint32_t yy = (y0 + row + 2 * a.ny - 1 - uint32_t(ey)) % a.ny;
        unit[n] = need ? (yy * a.nx + xx) | (s << 25) | (uint32_t(ez + 1) << 30) : ~0u;
    }
    const uint32_t wave_unit = __builtin_amdgcn_readfirstlane(tid & ~63u);

    auto wrapz = [&](int z) { return uint32_t(z < 0 ? z + int(a.nz) : z >= int(a.nz) ? z - int(a.nz) : z); };
    // sends plane p's sources on their way to the stage
    auto load_plane = [&](int p) {
        const uint32_t zp = wrapz(p);
        const uint32_t zn = wrapz(int(zp) + 1) * a.nxny, zc = zp * a.nxny, zl = wrapz(int(zp) - 1) * a.nxny;
#pragma unroll
        for (int n = 0; n < NI; ++n) {
            uint32_t v = unit[n];
            __asm__ volatile("" : "+v"(v));  // unpacked in every plane: hoisted, its parts take 3 registers
            const uint32_t ez1 = v >> 30;
            if (ez1 != 3u) {
                const uint32_t g = (v & 0x1FFFFFFu) + (ez1 == 0 ? zn : ez1 == 1 ? zc : zl);
                const uint32_t run = (g >> CB) * Q + ((v >> 25) & 31u);  // (chunk, direction) run of CH values
                const char *src = reinterpret_cast<const char *>(fin) + uint64_t(run) * (CH * kSize) +
                                  (g & (CH - 1u)) * kSize;
                load_lds(src, reinterpret_cast<char *>(stage) + (uint32_t(n) * BS + wave_unit) * 16);
            }
        }
    };

    T w[Q];
    each<0, Q>([&](auto s) { w[s] = S::weight(weight_class<L>(s), a); });
    st hold0[Q], up1[Q], up2[Q];  // arrivals waiting: e_z = 0 of plane p - 1, e_z = 1 of p - 1 and p - 2
    each<0, Q>([&](auto s) { hold0[s] = up1[s] = up2[s] = st(0); });
    auto update = [&](T (&f)[Q], int t, uint32_t g) {
        if constexpr (NET) {
            network_update<L, ST>(f, t, a, nullptr, w, g, &smlp, [] {});
        } else {
            T rho, ux, uy, uz;
            node_update<L, T, S::kShift, true, kConserve<ST, Q>, S::kScaled>(f, t, rho, ux, uy, uz, a, nullptr, w, g);
        }
    };
    int tn, tp = 0;
    load_plane(z0 - 1);
    tn = nd_type[wrapz(z0 - 1) * a.nxny + gxy];
    wait_vmcnt();
    for (int p = z0 - 1; p <= z1; ++p) {
        lds_barrier();  // plane p is staged; the last exchange has been read
        T f[Q];
        st o[Q];
        each<0, Q>([&](auto s) { o[s] = sp[s * (H * SW) - L::ex[s]]; });
        lds_barrier();  // ... and is in registers
        const int t = tn;
        if (p < z1) {
            load_plane(p + 1);
            tn = nd_type[wrapz(p + 1) * a.nxny + gxy];
        }
        each<0, Q>([&](auto s) { f[s] = S::in(o[s], s, a); });
        uint32_t g = wrapz(p) * a.nxny + gxy;
        update(f, t, g);
        each<0, Q>([&](auto s) { o[s] = S::step_out(f[s], s, a, 0u); });
        if (live) {
            each<0, Q>([&](auto s) {
                if constexpr (pair_moves<L>(s)) wp[pair_slot<L>(s) * (W * H)] = o[s];
            });
        }
        lds_barrier();  // the exchange is written
        if (wave_own) {
            if (own) {
                each<0, Q>([&](auto s) {
                    if constexpr (pair_moves<L>(s)) o[s] = wp[pair_slot<L>(s) * (W * H) - L::ey[s] * W - L::ex[s]];
                });
            }
            if (p > z0) {
                each<0, Q>([&](auto s) {
                    f[s] = S::in(L::ez[s] < 0 ? o[s] : L::ez[s] == 0 ? hold0[s] : up2[s], s, a);
                });
                g = uint32_t(p - 1) * a.nxny + gxy;
                update(f, tp, g);
                // the plane's first chunk by a descriptor, the rest by the lane
                const uint32_t first = uint32_t(p - 1) * a.nxny, c = first >> CB;
                const uint64_t back = uint64_t(c) * (Q * CH * kSize);
                const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(uintptr_t(fout) + back, a.fbytes - back);
                const uint32_t r = gxy + (first - c * CH);
                const uint32_t off = (r + __umul24(r >> CB, (Q - 1) * CH)) * kSize;
                wait_vmcnt();  // plane p + 1 has landed (ahead of the stores, which then need no count)
                if (own) {
                    each<0, Q>([&](auto s) {
                        RawBuf<st>::template store<kAuxNT>(S::step_out(f[s], s, a, 0u), rsrc, off,
                                                           uint32_t(s) * CH * kSize);
                    });
                }
            } else {
                wait_vmcnt();
            }
            each<0, Q>([&](auto s) {
                if constexpr (L::ez[s] == 0) hold0[s] = o[s];
                if constexpr (L::ez[s] > 0) { up2[s] = up1[s]; up1[s] = o[s]; }
            });
        } else {
            wait_vmcnt();
        }
        tp = t;
    }
}

}  // namespace tlbm

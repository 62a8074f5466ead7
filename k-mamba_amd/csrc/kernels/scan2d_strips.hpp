// scan2d_strips.hpp - the 2D recurrence on strips of rows, for the ScanND
// forward and for the backward's adjoint state.
//
//   s[p] = in[p] + e0 s[before p on axis 0] + e1 s[before p on axis 1]
//
// The grid's critical path is n0 + n1 - 1 points long, so what bounds a grid
// of few channel groups, or of small tiles handed over through memory, is the
// hand-over: a tile per wave with a flag in the L2 costs a store
// acknowledgement, a flag round trip and a load per tile (about 5.7 us per 8 x
// 4 tile). Here a workgroup takes a strip of kStripRows rows for one channel
// group (64 channel-states, one per lane): each compute wave owns a row and
// runs along it in blocks of kStripCols points, a few blocks behind the wave of
// the row before it, whose block it finds in an LDS ring (two LDS round trips
// per hand-over). Waves wait for each other through LDS counters only, never at
// a barrier, so one wave's memory latency does not stop the others, and the
// operands of kStripAhead blocks are in flight ahead of the arithmetic.
//
// Strips of one channel group are chained through the L2 of the XCD that owns
// the group (scannd_flow.hpp): wave 0, the courier, stores the strip's last
// row for the wave that computed it, waits for the L2's acknowledgement,
// publishes the block's flag, and in the other direction polls the previous
// strip's flags (64 blocks per load) and puts its last row into the first
// compute wave's ring. Having no other memory traffic it can wait for its
// stores without waiting for anyone's prefetched operands. A wait that runs
// out of polls feeds NaN to the first row instead, so every point that depends
// on the missing row is NaN, and sets the launch's status word.
//
// An item (strip, channel group) is taken from the XCD's queue in strip order
// by a running workgroup after the strip before it was taken: the waits end.
//
// Forward, M = 16 (tiles before -> strips): 64x64 D256 161 -> 95 us, 45x61 D96
// 125 -> 55, 12x250 D32 262 -> 53, 250x12 D32 156 -> 134 (36 strips in a
// chain), 17x19 D16 34.5 -> 17.4, 200x190 D48 399 -> 285; 256x256 D256, which
// fills the chip either way, 949 -> 870 (4.0 TB/s). Blocks in flight on the
// last two: 3: 300, 965; 4: 285, 870; 5: 287, 866; 6 (spills): 286, 877.
// Forward and backward, tiles in both -> strips in both: 45x61 D96 401 -> 150
// (221 with the forward's alone), 12x250 D48 719 -> 126, 30x24 D32 153 -> 80,
// 250x12 D48 381 -> 292, one row of 600 802 -> 102, one column of 600 568 -> 97.
#pragma once

#include <algorithm>
#include <utility>

#include "km_device.hpp"
#include "../km_runtime.hpp"
#include "scannd_flow.hpp"

namespace km {

constexpr int kStripWaves = 8;                    // the courier and one wave per row
constexpr int kStripRows = kStripWaves - 1;
constexpr int kStripCols = 4;
constexpr int kStripAhead = 4;                    // blocks of operands in flight
constexpr int kStripRing = 8;                     // blocks a ring holds

struct StripArgs {
    const float *u;            // [P, D] x (adjoint: dy)
    const float *B, *C;        // [P, D, M] (adjoint: C only)
    const float *dt0, *dt1;    // [P, D] per axis
    const float *A0, *A1;      // [D, M] per axis
    float *s;                  // [P, D, M] the states (adjoint: g)
    float *y;                  // [P, D] (forward)
    int n0, n1, D, DM, ncg, nblk, M;
};

__device__ __forceinline__ int strip_count(const int *p) {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ __forceinline__ void strip_set(int *p, int v) {
    if ((threadIdx.x & 63) == 0) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// The LDS serves a wave's accesses in order, so data before a counter's store,
// and after its load, needs the compiler's order only.
__device__ __forceinline__ void strip_order() { asm volatile("" ::: "memory"); }
// Until *p >= v; seen: the latest value read, which saves the LDS round trip
// while it suffices. The writer is a wave of this workgroup whose own waits
// end.
__device__ __forceinline__ void strip_wait(const int *p, int v, int &seen) {
    while (seen < v) {
        seen = strip_count(p);
        if (seen < v) __builtin_amdgcn_s_sleep(1);
    }
    strip_order();
}

// ADJ runs rows and columns backwards: strip 0 holds the last rows, block 0
// the last columns.
// MM: the M lanes of a channel (forward; the adjoint sums no lanes and takes
// any M).
template <int MM, bool ADJ>
__global__ void __launch_bounds__(64 * kStripWaves, 2) scan2d_strips(StripArgs p, FlowArgs f) {
    using F = bio<f32_t>;
    constexpr int CB = kStripCols, PF = kStripAhead, RG = kStripRing;
    constexpr unsigned kDrop = 0x80000000u;
    // ring[j]: blocks from wave j (0: the courier) to wave j + 1 (the last
    // row's to the courier).
    __shared__ __align__(16) float ring[kStripWaves][RG][64][CB];
    __shared__ int put[kStripWaves], got[kStripWaves];   // blocks written to / read from each ring
    __shared__ unsigned s_item;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
    const int xcd = flow_xcd();
    const int cg0 = f.cg_lo[xcd], ncx = f.cg_lo[xcd + 1] - cg0;
    if (ncx <= 0) return;
    const int nstrip = (p.n0 + kStripRows - 1) / kStripRows, nb = p.nblk;
    const unsigned nitems = static_cast<unsigned>(nstrip) * static_cast<unsigned>(ncx);
    const unsigned epoch = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(f.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    const float qnan = __builtin_nanf("");
    for (;;) {
        __syncthreads();                          // the previous item's counters are read
        if (threadIdx.x == 0) s_item = atomicAdd(&f.counter[xcd], 1u);
        if (threadIdx.x < kStripWaves) {
            put[threadIdx.x] = 0;
            got[threadIdx.x] = 0;
        }
        __syncthreads();
        const unsigned item = __builtin_amdgcn_readfirstlane(s_item);
        if (item >= nitems) break;
        const int strip = static_cast<int>(item / ncx), cg = cg0 + static_cast<int>(item % ncx);
        const int fl = cg * 64 + lane;            // this lane's channel-state
        const int d = ADJ ? fl / p.M : fl / MM;
        const int vf = fl * 4, vd = d * 4;
        const int i0 = strip * kStripRows;        // the strip's first row, in walking order
        const int nrow = min(kStripRows, p.n0 - i0);
        const bool feeds = strip + 1 < nstrip;    // another strip needs the last row
        auto row_of = [&](int i) { return ADJ ? p.n0 - 1 - i : i; };
        auto win = [](long b) { return b < 0x7fffffffL ? b : 0x7fffffffL; };
        auto rsrc_s = [&](int i) {
            return make_rsrc(p.s + static_cast<long>(row_of(i)) * p.n1 * p.DM, win(static_cast<long>(p.n1) * p.DM * 4));
        };
        // Column c of block k: blocks cover [4 b, 4 b + 4), b descending for ADJ.
        auto blk = [&](int k) { return ADJ ? nb - 1 - k : k; };
        unsigned *const fbase = f.flags + (static_cast<long>(strip) * p.ncg + cg) * nb;   // [block]

        if (w == 0) {
            // ---- the courier -----------------------------------------------
            const int nin = strip > 0 ? nb : 0, nout = feeds ? nb : 0;
            const auto rin = rsrc_s(strip > 0 ? i0 - 1 : i0), rout = rsrc_s(i0 + nrow - 1);
            const unsigned *fin = fbase - static_cast<long>(p.ncg) * nb;   // the previous strip's (strip > 0)
            int din = 0, dout = 0;
            unsigned idle = 0;
            bool lost = false;
            while (din < nin || dout < nout) {
                // The last row's new blocks to memory.
                const int have = nout > 0 ? strip_count(&put[nrow]) : 0;
                strip_order();
                const int take = min(have - dout, 4);
                for (int q = 0; q < take; ++q) {
                    const int b = blk(dout + q);
#pragma unroll
                    for (int c = 0; c < CB; ++c) {
                        const int col = b * CB + c;
                        const float v = ring[nrow][(dout + q) % RG][lane][c];
                        F::st(rout, static_cast<int>(col < p.n1 ? static_cast<unsigned>(vf) : kDrop),
                              min(col, p.n1 - 1) * p.DM * 4, v);
                    }
                }
                // The previous strip's flags from block din on.
                const int space = nin > 0 ? RG - (din - strip_count(&got[0])) : 0;
                strip_order();
                int ready = 0;
                const bool ask = din < nin && space > 0;
                if (ask && !lost) {
                    if (idle >= f.spin) {
                        lost = true;
                        if (lane == 0) __hip_atomic_store(f.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    } else {
                        bool ok = false;
                        if (din + lane < nin)
                            ok = __hip_atomic_load(fin + din + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch;
                        const unsigned long long m = __ballot(ok);
                        ready = ~m == 0 ? 64 : __builtin_ctzll(~m);
                        if (ready == 0) ++idle;
                        else idle = 0;
                    }
                }
                if (ask && lost) ready = nin - din;
                const int n = min(min(ready, space), 4);
                if (take > 0) {
                    __builtin_amdgcn_s_waitcnt(0);   // this wave's stores acknowledged by the L2
                    if (lane < take)
                        __hip_atomic_store(fbase + dout + lane, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    dout += take;
                    strip_set(&got[nrow], dout);
                }
                for (int q = 0; q < n; ++q) {
                    const int b = blk(din + q);
                    float v[CB];
#pragma unroll
                    for (int c = 0; c < CB; ++c)
                        v[c] = lost ? qnan : F::ld_agent(rin, vf, min(b * CB + c, p.n1 - 1) * p.DM * 4);
#pragma unroll
                    for (int c = 0; c < CB; ++c) ring[0][(din + q) % RG][lane][c] = v[c];
                }
                if (n > 0) {
                    strip_order();
                    din += n;
                    strip_set(&put[0], din);
                }
                if (n == 0 && take <= 0) __builtin_amdgcn_s_sleep(1);
            }
            continue;
        }

        // ---- a row -----------------------------------------------------------
        if (w > nrow) continue;
        const int i = i0 + w - 1, r = row_of(i);
        const bool from = i > 0;                        // a row before this one
        const bool to_ring = w < nrow || feeds;         // the next wave, or the courier, reads this row
        const bool store = w < nrow || !feeds;          // else the courier stores it
        const long row_d = static_cast<long>(r) * p.n1 * p.D, row_s = static_cast<long>(r) * p.n1 * p.DM;
        // Pointers to the block that is loaded next and to the one that is
        // stored next, moved by a block at a time (scalar adds).
        const long first_d = row_d + static_cast<long>(blk(0)) * CB * p.D;
        const long first_s = row_s + static_cast<long>(blk(0)) * CB * p.DM;
        const long step_d = static_cast<long>(ADJ ? -CB : CB) * p.D, step_s = static_cast<long>(ADJ ? -CB : CB) * p.DM;
        const float *pu = p.u + first_d;
        // The adjoint's axis-0 decay is that of the point it flows from.
        const float *pd0 = p.dt0 + first_d + (ADJ && from ? static_cast<long>(p.n1) * p.D : 0);
        const float *pdt1 = p.dt1 + first_d;
        const float *pb = (ADJ ? p.C : p.B) + first_s, *pc = p.C + first_s;
        float *ps = p.s + first_s, *py = ADJ ? nullptr : p.y + first_d;
        const float A0 = p.A0[fl] * kLog2e, A1 = p.A1[fl] * kLog2e;
        // Lane offsets of a block's columns; the block's first column is in the
        // resources' base, and their size ends at the row's end: columns past
        // it load 0 and their stores are dropped, with no select.
        unsigned od[CB], om[CB];
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            od[c] = static_cast<unsigned>(vd + c * p.D * 4);
            om[c] = static_cast<unsigned>(vf + c * p.DM * 4);
        }
        // M = 16: the four columns' readouts are scattered over a channel's 16
        // lanes (row_readout): one y store a block.
        constexpr bool kRowY = MM == 16;
        const unsigned oy = static_cast<unsigned>(kRowY ? (((lane % 16) / 4) * p.D + d) * 4 : vd);
        const bool ylane = kRowY ? lane % 4 == 0 : lane % MM == 0;
        // (A dropped offset keeps its bit 31 with a column's offset added.)
        const unsigned ydrop = ylane ? 0u : kDrop, sdrop = store ? 0u : kDrop;
        struct Ops {
            float u[CB], d0[CB], d1[CB], b[CB], c[CB];
        };
        auto load = [&](int k, Ops &o) __attribute__((always_inline)) {
            // (Blocks past the last one are of size 0: their loads are not made.)
            const int left = k < nb ? p.n1 - blk(k) * CB : 0;
            const int nd = left * p.D * 4, nm = left * p.DM * 4;
            const auto ru = make_rsrc(pu, nd), rd0 = make_rsrc(pd0, nd), rd1 = make_rsrc(pdt1, nd);
            const auto rB = make_rsrc(pb, nm), rC = make_rsrc(pc, nm);
            pu += step_d;
            pd0 += step_d;
            pdt1 += step_d;
            pb += step_s;
            if constexpr (!ADJ) pc += step_s;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                o.u[c] = F::ld(ru, static_cast<int>(od[c]), 0);
                o.d0[c] = F::ld(rd0, static_cast<int>(od[c]), 0);
                o.d1[c] = F::ld(rd1, static_cast<int>(od[c]), 0);
                o.b[c] = F::ld(rB, static_cast<int>(om[c]), 0);
                if constexpr (!ADJ) o.c[c] = F::ld(rC, static_cast<int>(om[c]), 0);
            }
        };
        float prev = 0.f, pd1 = 0.f;        // the neighbour on axis 1 (and, ADJ, its delta)
        int seen_in = 0, seen_out = 0;
        auto block = [&](int k, Ops &o) __attribute__((always_inline)) {
            const int col0 = blk(k) * CB;
            float e0[CB], e1[CB], in[CB];
            // What does not depend on a neighbour, before the wait for one.
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                e0[c] = exp2_fast(o.d0[c] * A0);
                e1[c] = exp2_fast(o.d1[c] * A1);
                in[c] = ADJ ? o.u[c] * o.b[c] : ((o.d0[c] + o.d1[c]) * 0.5f) * (o.b[c] * o.u[c]);
            }
            if (from) {
                strip_wait(&put[w - 1], k + 1, seen_in);
                float top[CB];
#pragma unroll
                for (int c = 0; c < CB; ++c) top[c] = ring[w - 1][k % RG][lane][c];
                strip_order();
                strip_set(&got[w - 1], k + 1);   // in order after the reads
#pragma unroll
                for (int c = 0; c < CB; ++c) in[c] = fmaf(e0[c], top[c], in[c]);
            }
            float out[CB];
            if constexpr (ADJ) {
                // The row's last block comes first: its columns past the end
                // are skipped, its last one has no successor.
#pragma unroll
                for (int c = CB - 1; c >= 0; --c) {
                    const bool succ = k > 0 || col0 + c + 1 < p.n1, live = k > 0 || col0 + c < p.n1;
                    out[c] = succ ? fmaf(pd1, prev, in[c]) : in[c];
                    prev = live ? out[c] : prev;
                    pd1 = live ? e1[c] : pd1;      // the decay from this column to the next
                }
            } else {
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    out[c] = (c > 0 || k > 0) ? fmaf(e1[c], prev, in[c]) : in[c];
                    prev = out[c];
                }
            }
            if (to_ring) {
                strip_wait(&got[w], k - RG + 1, seen_out);
#pragma unroll
                for (int c = 0; c < CB; ++c) ring[w][k % RG][lane][c] = out[c];
                strip_order();
                strip_set(&put[w], k + 1);
            }
            const auto rs = make_rsrc(ps, (p.n1 - col0) * p.DM * 4);
            ps += step_s;
#pragma unroll
            for (int c = 0; c < CB; ++c) F::st(rs, static_cast<int>(om[c] | sdrop), 0, out[c]);
            if constexpr (!ADJ) {
                const auto ry = make_rsrc(py, (p.n1 - col0) * p.D * 4);
                py += step_d;
                float yr[CB];
#pragma unroll
                for (int c = 0; c < CB; ++c) yr[c] = o.c[c] * out[c];
                if constexpr (kRowY) {
                    F::st(ry, static_cast<int>(oy | ydrop), 0, row_readout<CB>(yr));
                } else {
#pragma unroll
                    for (int c = 0; c < CB; ++c)
                        F::st(ry, static_cast<int>((oy + c * p.D * 4) | ydrop), 0, sum_m_lanes<MM>(yr[c]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            load(k + PF, o);
            __builtin_amdgcn_sched_barrier(0);
        };
        Ops q[PF];
#pragma unroll
        for (int u = 0; u < PF; ++u) load(u, q[u]);
        // Whole groups without a branch around the loads: a branch would make
        // the compiler wait for more of them at its join.
        int k = 0;
        for (; k + PF <= nb; k += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u) block(k + u, q[u]);
        }
#pragma unroll
        for (int u = 0; u < PF - 1; ++u)
            if (k + u < nb) block(k + u, q[u]);
    }
}

// Flags a strip launch needs, and whether the kernel's 32-bit row offsets
// cover the grid.
inline long strip_flags(long n0, long n1, long ncg) {
    return ((n0 + kStripRows - 1) / kStripRows) * ((n1 + kStripCols - 1) / kStripCols) * ncg;
}
inline bool strip_fits(long n0, long n1, long DM) {
    return DM % 64 == 0 && ((n1 == 1 ? n0 : n1) + kStripCols) * DM * 4 < 0x7fffffffL &&
           strip_flags(n0, n1, DM / 64) < 0x7fffffffL;
}

// The launch: up to one workgroup per CU of an XCD (their registers allow no
// more). A grid of one column is one row with the axes exchanged: a single
// strip (which uses no flag) instead of a chain of them.
template <bool ADJ>
static int launch_strips(StripArgs a, const FlowArgs &fa, hipStream_t s) {
    if (a.n1 == 1) {
        std::swap(a.n0, a.n1);
        std::swap(a.dt0, a.dt1);
        std::swap(a.A0, a.A1);
        a.nblk = (a.n1 + kStripCols - 1) / kStripCols;
    }
    const long nstrip = (a.n0 + kStripRows - 1) / kStripRows;
    long per_xcd = 0;
    for (int x = 0; x < 8; ++x) per_xcd = std::max<long>(per_xcd, nstrip * (fa.cg_lo[x + 1] - fa.cg_lo[x]));
    const dim3 grid(static_cast<unsigned>(8 * std::min<long>(per_xcd, 32))), blk(64 * kStripWaves);
#define KM_STRIP(MMv) hipLaunchKernelGGL((scan2d_strips<MMv, ADJ>), grid, blk, 0, s, a, fa)
    switch (ADJ ? 1 : a.M) {
    case 1: KM_STRIP(1); break;
    case 2: KM_STRIP(ADJ ? 1 : 2); break;
    case 4: KM_STRIP(ADJ ? 1 : 4); break;
    case 8: KM_STRIP(ADJ ? 1 : 8); break;
    case 16: KM_STRIP(ADJ ? 1 : 16); break;
    case 32: KM_STRIP(ADJ ? 1 : 32); break;
    default: KM_STRIP(ADJ ? 1 : 64); break;
    }
#undef KM_STRIP
    KM_HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace km

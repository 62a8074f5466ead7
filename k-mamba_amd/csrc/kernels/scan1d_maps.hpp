// scan1d_maps.hpp - the map pass of a Scan1D sequence split over workgroups.
//
// Over a run of steps the recurrence is an affine map of the state that
// enters it: h -> exp(A * sum delta) h + h_end with h_end the state that the
// steps reach from zero, and the adjoint, run backwards, is the same with
// g_end. The map pass finds (h_end, sum delta) of parts of Lm steps; the pass
// that produces the outputs then starts every segment at once, each from the
// state it folds from the maps before (adjoint: after) it.
#pragma once

#include <algorithm>
#include <type_traits>

#include "km_device.hpp"
#include "../km_runtime.hpp"

namespace km {

// The windowed kernels address B / C by rows of bc_st elements and read 0 past a
// batch element's L rows, so a row must hold every channel's states. Other
// strides (channel-major [D, L, N], B / C constant over time) go to the
// sequential kernels.
inline bool rows_hold_channels(long D, long N, long st, long sd) { return (D - 1) * sd + N <= st; }

// A fold of maps takes h to 2^z h + add from map to map, z the exponent of the
// decay over the map's steps, which may be out of range by itself: with 2^z =
// inf a state of exactly 0 (padded x, masked dy) becomes NaN, with 2^z = 0 an
// infinite one. An overflow anywhere leaves the fold's result infinite or NaN
// in some lane; then it is run again with decay_add, where the integer part of
// z goes to h's exponent, so that a product is in range where the steps' own
// products are. (decay_add in every fold takes 1 us of the 72 us of B1 L5003
// D1536 bf16 gated; the check 0.2.)
__device__ __forceinline__ bool fold_overflowed(float h) { return __any(!(fabsf(h) < __builtin_inff())); }
__device__ __forceinline__ float decay_add(float z, float h, float add) {
    const float k = fminf(fmaxf(floorf(z), -1e9f), 1e9f);
    return fmaf(exp2_fast(z - k), __builtin_amdgcn_ldexpf(h, static_cast<int>(k)), add);
}

struct MapArgs {
    const void *x;         // [B, L, D] the forward's x, the adjoint's dy
    const void *dt;        // [B, L, D]
    const void *M;         // the forward's B, the adjoint's C (strides sb, st, sd)
    const float *A;        // [D, 16]
    long L, D, sb, st, sd;
    int nmap, Lm;          // parts per sequence and steps per part
    int t0;                // first step of part 0; parts end at L at the latest
    float *seg_h;          // [B, nmap, D, 16] end states from zero
    float *seg_dsum;       // [B, nmap, D] sums of delta
    // Forward: clamp flags of the replay's 32-channel groups to clear, and a
    // copy of h0 [B, D, 16] where h_final shares h0's memory (the last
    // segment's replay writes it while earlier ones may not have started);
    // each or null.
    int *clamp_flag;
    const float *h0;
    float *h0_copy;
};

// Only the end state is wanted, so there is nothing to replay and no carry
// to pass along: each of the workgroup's 8 waves runs its own eighth of the
// part from zero without a barrier, and the 8 maps are composed once at the
// end. A lane owns a whole channel (all 16 states), which halves the work per
// step that does not depend on the state (exp, delta * x, addresses) against
// the output pass's two or four lanes per channel. Bound by VALU issue (decay,
// input and FMA: 3 of ~3.8 instructions per state update): forward, B1 L4992
// D1536 bf16 in 5 segments, whole call 79.2 -> 72.4 us against a map pass
// that ran the output kernel's local passes and folds. kMapBlock rows of x,
// delta and M are in flight ahead of the arithmetic; the wave's M rows go
// through its own LDS rows, from which every lane reads the same 16 values.
constexpr int kMapWaves = 8, kMapBlock = 8;
// VEC (per-channel M, whose loads bound the pass): a lane's 16 states in 16-byte
// loads. B1 L16384 D64 bf16, whole call: 145 us, with 16 loads of 2 bytes 250,
// with the output kernel as the map pass 194.
template <typename T, bool SHARED, bool ADJ, bool VEC>
__global__ void __launch_bounds__(64 * kMapWaves, 4) scan1d_segment_map(MapArgs p) {
    using IO = bio<T>;
    constexpr int N = 16, TS = IO::size, MB = kMapBlock, W = kMapWaves, PADC = 65;
    // Staged M rows of each wave (two blocks), then the waves' end states
    // [wave][state][channel] (rows padded against bank conflicts).
    __shared__ __align__(16) float lds[W * N * PADC];
    __shared__ float sds[W][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned ngroups = static_cast<unsigned>((p.D + 63) / 64);
    const unsigned wg = static_cast<unsigned>(xcd_remap(blockIdx.x, gridDim.x));
    const unsigned bs = wg / ngroups, grp = wg - bs * ngroups;
    const unsigned nmap = static_cast<unsigned>(p.nmap);
    const long b = bs / nmap;
    const unsigned part = bs - static_cast<unsigned>(b) * nmap;
    const long d0 = static_cast<long>(grp) * 64, d = d0 + lane;
    const bool dvalid = d < p.D;
    const long dc = dvalid ? d : p.D - 1;
    // This wave's steps [ta, ta + nt) of the sequence; the last parts may be
    // short or empty (identity maps).
    const long pa = p.t0 + static_cast<long>(part) * p.Lm;
    const int len = static_cast<int>(max(0L, min(static_cast<long>(p.Lm), p.L - pa)));
    const int q = (p.Lm + W - 1) / W;
    const int wa = min(w * q, len), nt = min(q, len - wa);
    const long ta = min(pa + wa, p.L);
    const long row0 = b * p.L + ta;
    const auto rx = make_rsrc(static_cast<const char *>(p.x) + row0 * p.D * TS, static_cast<long>(nt) * p.D * TS);
    const auto rdt = make_rsrc(static_cast<const char *>(p.dt) + row0 * p.D * TS, static_cast<long>(nt) * p.D * TS);
    const long m0 = b * p.sb + ta * p.st;
    const auto rM = make_rsrc(static_cast<const char *>(p.M) + m0 * TS, static_cast<long>(nt) * p.st * TS);
    const int rowx = static_cast<int>(p.D) * TS, rowm = static_cast<int>(p.st) * TS;
    const int vx = static_cast<int>(dc) * TS;
    const int vm = SHARED ? (lane & 15) * TS : static_cast<int>(dc * p.sd) * TS;
    // Row i of the wave's walk: step ta + i, from the last step down for the
    // adjoint (a row past the end, or before step 0 whose offset is negative
    // and so past the window, reads as 0: an identity step).
    auto row = [&](int i) { return ADJ ? nt - 1 - i : i; };

    float X[MB], Dl[MB], rb[2];
    auto load = [&](int i, float (&xo)[MB], float (&dlo)[MB]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < MB; ++k) {
            xo[k] = IO::ld(rx, vx + row(i + k) * rowx, 0);
            dlo[k] = IO::ld(rdt, vx + row(i + k) * rowx, 0);
        }
        if constexpr (SHARED) {
#pragma unroll
            for (int u = 0; u < 2; ++u) rb[u] = IO::ld(rM, vm + row(i + 4 * u + (lane >> 4)) * rowm, 0);
        }
    };
    load(0, X, Dl);
    // Decays of this lane's channel, exp2(delta * A log2 e), and whether every
    // channel of the workgroup has A[d, n] = (n + 1) A[d, 0].
    float Ap[N];
    bool structured = true;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const float a = p.A[dc * N + n];
        structured = structured && a == static_cast<float>(n + 1) * p.A[dc * N];
        Ap[n] = a * kLog2e;
    }
    const bool fast = __builtin_amdgcn_readfirstlane(__syncthreads_and(structured)) != 0;
    // The powers e1^(n+1) as products of two lower ones (log-depth).
    auto powers = [&](float e1, float (&e)[N]) __attribute__((always_inline)) {
        e[0] = e1;
#pragma unroll
        for (int n = 1; n < N; ++n) e[n] = e[(n - 1) / 2] * e[n - 1 - (n - 1) / 2];
    };
    float h[N], dsum = 0.f;
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = 0.f;
    float *const rows = lds + w * (2 * MB * N);
    auto sweep = [&](auto fastc) __attribute__((always_inline)) {
        constexpr bool FAST = decltype(fastc)::value;
        for (int t = 0, buf = 0; t < nt; t += MB, buf ^= 1) {
            float *const tile = rows + buf * (MB * N);
            if constexpr (SHARED) {
                tile[lane] = rb[0];
                tile[64 + lane] = rb[1];
            }
            float xs[MB], ds[MB];
#pragma unroll
            for (int k = 0; k < MB; ++k) {
                xs[k] = X[k];
                ds[k] = Dl[k];
            }
            load(t + MB, X, Dl);
            __builtin_amdgcn_wave_barrier();      // the rows are this wave's own: LDS order suffices
#pragma unroll
            for (int k = 0; k < MB; ++k) {
                float mv[N];
                if constexpr (VEC) {
                    IO::ld16(rM, vm + row(t + k) * rowm, mv);
                } else {
#pragma unroll
                    for (int n = 0; n < N; ++n)
                        mv[n] = SHARED ? tile[k * N + n] : IO::ld(rM, vm + n * TS + row(t + k) * rowm, 0);
                }
                const float u = ADJ ? xs[k] : ds[k] * xs[k];
                dsum += ds[k];
                float e[N];
                if constexpr (FAST) {
                    powers(exp2_fast(ds[k] * Ap[0]), e);
                } else {
#pragma unroll
                    for (int n = 0; n < N; ++n) e[n] = exp2_fast(ds[k] * Ap[n]);
                }
#pragma unroll
                for (int n = 0; n < N; ++n)
                    h[n] = ADJ ? fmaf(u, mv[n], h[n]) * e[n] : fmaf(e[n], h[n], mv[n] * u);
            }
        }
    };
    if (fast) sweep(std::true_type{});
    else sweep(std::false_type{});
    __syncthreads();                               // the staged rows are read; their memory is reused
    sds[w][lane] = dsum;
#pragma unroll
    for (int n = 0; n < N; ++n) lds[(w * N + n) * PADC + lane] = h[n];
    __syncthreads();
    // Compose the waves' maps in the order of the walk: state i % 16 of
    // channel i / 16 by thread i (and i + 512), so the stores are contiguous.
#pragma unroll
    for (int i = tid; i < 64 * N; i += 64 * W) {
        const int n = i & 15, c = i >> 4;
        const long dd = d0 + c;
        if (dd < p.D) {
            const float a2 = p.A[dd * N + n] * kLog2e;
            float run = 0.f;
#pragma unroll
            for (int u = 0; u < W; ++u) {
                const int v = ADJ ? W - 1 - u : u;
                run = fmaf(exp2_fast(sds[v][c] * a2), run, lds[(v * N + n) * PADC + c]);
            }
            if (fold_overflowed(run)) {
                run = 0.f;
#pragma unroll 1
                for (int u = 0; u < W; ++u) {
                    const int v = ADJ ? W - 1 - u : u;
                    run = decay_add(sds[v][c] * a2, run, lds[(v * N + n) * PADC + c]);
                }
            }
            p.seg_h[(static_cast<long>(bs) * p.D + dd) * N + n] = run;
            if (!ADJ && part == 0 && p.h0_copy)
                p.h0_copy[(b * p.D + dd) * N + n] = p.h0[(b * p.D + dd) * N + n];
        }
    }
    if (w == 0 && dvalid) {
        float tot = 0.f;
#pragma unroll
        for (int v = 0; v < W; ++v) tot += sds[v][lane];
        p.seg_dsum[static_cast<long>(bs) * p.D + d] = tot;
    }
    if (!ADJ && p.clamp_flag && part == 0 && tid < 2 && d0 + 32 * tid < p.D)
        p.clamp_flag[b * ((p.D + 31) / 32) + 2 * static_cast<long>(grp) + tid] = 0;
}

// Parts per segment of Ls steps (a multiple of 64) for maps of nsegs
// segments: 1, 2, 4 or 8, the first that gives the map pass a workgroup (64
// channels) per CU, with at most kMaxMaps maps for a fold.
constexpr long kMaxMaps = 64;
inline long map_parts(long B, long D, long nsegs, long Ls) {
    const long groups = (D + 63) / 64;
    long r = 1;
    while (r < 8 && B * groups * nsegs * r < 256 && nsegs * r * 2 <= kMaxMaps && Ls / (2 * r) >= 64) r *= 2;
    return r;
}

template <typename T, bool ADJ>
static int launch_maps(const MapArgs &m, long B, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(B * m.nmap * ((m.D + 63) / 64))), blk(64 * kMapWaves);
    // The loads' dwords have to be aligned, which 4-byte elements are.
    constexpr uintptr_t es = bio<T>::size;
    const bool dwords = ((reinterpret_cast<uintptr_t>(m.M) | m.sb * es | m.st * es | m.sd * es) & 3) == 0;
    if (m.sd == 0)   hipLaunchKernelGGL((scan1d_segment_map<T, true, ADJ, false>), grid, blk, 0, s, m);
    else if (dwords) hipLaunchKernelGGL((scan1d_segment_map<T, false, ADJ, true>), grid, blk, 0, s, m);
    else             hipLaunchKernelGGL((scan1d_segment_map<T, false, ADJ, false>), grid, blk, 0, s, m);
    KM_HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace km

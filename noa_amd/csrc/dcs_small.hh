// Maps too small to fill the chip with one lane per pair: one workgroup per
// 64 pairs, the integrals spread over lanes by quadrature node.
//
// What bounds a small map is the length of one wave's instruction chain (a
// closed form, then up to 9 photonuclear nodes of ~470 FP64 instructions
// each), not the chip: 10,000 pairs in tiles of 2048 are 5 workgroups on 256
// CUs and took 88 us, in tiles of 256 pairs 26 us. Here the four waves of a
// workgroup share 64 pairs:
//   1. wave 0 evaluates bremsstrahlung and wave 1 ionisation, wave 2 runs
//      pair production's exit and its integral's set-up, wave 3 the same for
//      photonuclear; pairs whose integral runs become entries in LDS;
//   2. the nodes of all entries are work items (9 per photonuclear entry, 8
//      per pair-production one, whole waves of one kind): one or two chains
//      of a single node per wave instead of 9 in a row;
//   3. one lane per entry adds its nodes' terms in the serial loop's order
//      and finishes the pair, so the results equal the tile kernel's bit for
//      bit.
// Measured on MI355X, FP64, all four processes: 8.5 us for 256 to 16,384
// pairs (25-88 us in tiles of 2048), 14.4 us for 65,536 (88), 22 us for
// 131,072 (91; 30 in tiles of 256). A chain per node spends more on set-up
// (constants, LDS reads, partly filled waves), so per pair it is at ~65% of
// the tile kernel's speed once the chip is full: see eval_tile for the line.
// Larger groups (128 pairs) were 10% slower at 10,000 and 65,536 pairs. Built
// to 128 registers, four waves per SIMD; allowed more it takes 133, and three
// waves take 15.9 us for 65,536 pairs where four take 12.1 (a call into new
// tensors).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dcs_consts.hh"
#include "dcs_f64.hh"
#include "dcs_tile.hh"
#include "fastmath.hh"

namespace noa_hip {

constexpr int SMALL_TILE = 64;

// The open integrals of the 64 pairs: what an entry's nodes share, and the
// node terms. Entry e is the e-th pair (in tile order) whose integral runs.
struct SmallLds {
    double x8[8], w8[8], x9[9], w9[9];
    double pair_K[SMALL_TILE], pair_q[SMALL_TILE], pair_beta[SMALL_TILE], pair_tmin[SMALL_TILE];
    double pair_a[8 * SMALL_TILE], pair_b[8 * SMALL_TILE];
    double photo_K[SMALL_TILE];
    F64::PhotoPre photo[SMALL_TILE];
    double photo_f[9 * SMALL_TILE];
    uint8_t pair_at[SMALL_TILE], photo_at[SMALL_TILE];
    uint32_t n_pair, n_photo;
};

// Rank of this lane among the wave's lanes with pred set; *count their number.
__device__ __forceinline__ uint32_t wave_rank(bool pred, uint32_t* count) {
    const unsigned long long m = __ballot(pred);
    *count = uint32_t(__popcll(m));
    return __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
}

// Pairs [base, end), at most SMALL_TILE of them, by one workgroup. FP64
// physics for both output types: the mixed-precision form at these sizes is
// no faster in FP32, and its results are then the rounded FP64 values.
template <class OutT>
__device__ __forceinline__ void run_small(int64_t base, int64_t end, const double* __restrict__ K,
                                          const double* __restrict__ q, ConstsPtr cp, const Outs<OutT>& o,
                                          SmallLds& s, double* fm_block) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const fm::Tab t = fm::tab_from_block(fm_block);
    const int64_t g = base + lane;
    const bool valid = g < end;
    const double k = valid ? K[g] : 1., qq = valid ? q[g] : 0.;
    load_fm_tables(fm_block);
    if (threadIdx.x < 9) {  // the node tables in LDS: the node index varies by lane
        s.x9[threadIdx.x] = GL9_X[threadIdx.x];
        s.w9[threadIdx.x] = GL9_W[threadIdx.x];
        if (threadIdx.x < 8) {
            s.x8[threadIdx.x] = GL8_X[threadIdx.x];
            s.w8[threadIdx.x] = GL8_W[threadIdx.x];
        }
    }
    __syncthreads();
    const DcsConsts& c = item_consts(cp);
    // (entries hold fast-path pairs only, as F64::pair_at and F64::photo
    // select them; the few others are evaluated in their lane at once)
    const bool fast = c.fast_ok && k + c.mass <= F64::FAST_E_MAX;
    if (wave == 0) {
        if (valid && o.b) o.b[g] = OutT(F64::brems(k, qq, c, t));
    } else if (wave == 1) {
        if (valid && o.i) o.i[g] = OutT(F64::ion(k, qq, c, t));
    } else if (wave == 2) {
        uint32_t count = 0;
        if (o.p) {
            double argmin = 0.;
            const bool on = valid && F64::pair_active(k, qq, c, argmin);
            const uint32_t e = wave_rank(on && fast, &count);
            if (on && fast) {
                double gamma;
                const F64::PairPre p = F64::pair_setup<false, true, true>(k, qq, c, t, argmin, gamma);
                s.pair_K[e] = k;
                s.pair_q[e] = qq;
                s.pair_beta[e] = p.beta;
                s.pair_tmin[e] = p.tmin;
                s.pair_at[e] = uint8_t(lane);
            } else if (valid) {
                o.p[g] = OutT(on ? F64::pair_at(k, qq, argmin, c, t) : 0.);
            }
        }
        if (lane == 0) s.n_pair = count;
    } else {
        uint32_t count = 0;
        if (o.ph) {
            const bool on = valid && F64::photo_active(k, qq, c);
            const uint32_t e = wave_rank(on && fast, &count);
            if (on && fast) {
                s.photo[e] = F64::photo_setup<false, true>(k, qq, c, t);
                s.photo_K[e] = k;
                s.photo_at[e] = uint8_t(lane);
            } else if (valid) {
                o.ph[g] = OutT(on ? F64::photo(k, qq, c, t) : 0.);
            }
        }
        if (lane == 0) s.n_photo = count;
    }
    __syncthreads();
    const uint32_t nph = s.n_photo, npa = s.n_pair;
    const uint32_t wph = (nph * 9 + 63) / 64, tasks = wph + (npa * 8 + 63) / 64;
    for (uint32_t task = wave; task < tasks; task += WG / 64) {
        const DcsConsts& cn = item_consts(cp);
        if (task < wph) {
            const uint32_t v = task * 64 + lane;
            if (v < nph * 9) {
                const uint32_t e = v / 9, j = v - 9 * e;
                const F64::PhotoPre p = s.photo[e];
                s.photo_f[v] = F64::photo_node<false, true>(p, s.x9[j], cn, t);
            }
        } else {
            const uint32_t v = (task - wph) * 64 + lane;
            if (v < npa * 8) {
                const uint32_t e = v / 8, j = v % 8;
                const F64::PairPre p = F64::pair_pre(s.pair_q[e], s.pair_beta[e], s.pair_tmin[e], cn);
                double a, b;
                F64::pair_node<false, true>(p, s.x8[j], s.w8[j], cn, t, a, b);
                s.pair_a[v] = a;
                s.pair_b[v] = b;
            }
        }
    }
    __syncthreads();
    if (wave == 2 && uint32_t(lane) < npa) {
        double I = 0.;
        for (int j = 0; j < 8; j++) I = F64::pair_add<false>(s.pair_a[8 * lane + j], s.pair_b[8 * lane + j], I);
        const double pk = s.pair_K[lane];
        o.p[base + s.pair_at[lane]] = OutT(F64::pair_finish<false, true>(
            pk, s.pair_q[lane], F64::pair_gamma<true>(pk, c), s.pair_tmin[lane], I, c, t));
    } else if (wave == 3 && uint32_t(lane) < nph) {
        double ds = 0.;
        for (int j = 0; j < 9; j++) ds = F64::photo_add<false>(s.photo_f[9 * lane + j], s.w9[j], ds);
        o.ph[base + s.photo_at[lane]] =
            OutT(F64::photo_finish<false, true>(s.photo_K[lane], s.photo[lane], ds, c));
    }
}

template <class OutT>
__global__ __launch_bounds__(WG) void dcs_small_kernel(const double* __restrict__ K, const double* __restrict__ q,
                                                       int64_t n, DcsConsts, Outs<OutT> o) {
    __shared__ SmallLds s;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];
    run_small<OutT>(int64_t(blockIdx.x) * SMALL_TILE, n, K, q, kernarg_consts(), o, s, fm_block);
}

}  // namespace noa_hip

// Single-element DCS evaluation: FP64 and mixed FP32 kernels, the seeded
// workload generator, and their C entry points (include/noa_dcs.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "capi_util.hh"
#include "dcs_consts.hh"
#include "dcs_f32m.hh"
#include "dcs_f64.hh"
#include "dcs_small.hh"
#include "dcs_tile.hh"

namespace noa_hip {

// Pairs per workgroup of a map of n pairs: 64 is the small-map kernel
// (dcs_small.hh), larger ones the tile kernel below, whose tiles shorten from
// this towards the end of the map (TileCut). Four workgroups of the tile
// kernel fit a CU, 1024 the chip, and a tile of 2048 pairs among four lasts
// 150 us: below 1.5e6 pairs it would outlast the rest. Measured on MI355X
// (FP64 / mixed, us, at tiles of 64, 256, 1024, 2048):
//   131,072 pairs    22  30   -   -   /   22  33   -   -
//   250,000          41  38  43  42   /   41  39  43  43
//   414,000           -  59  59  60   /    -  55  55  55
//   600,000           -  76  64  64   /    -  68  58  58
//   1,240,000         - 137 115 118   /    - 119  97  95
//   3,000,017         -   - 234 233   /    -   - 188 181
//   8,000,000         -   - 583 565   /    -   - 450 419
//   16,777,216        -   - 1196 1168 /    -   - 912 844
inline int eval_tile(int64_t n) {
    if (n <= 200000) return 64;
    if (n <= 300000) return 256;
    if (n <= 1500000) return 1024;
    return 2048;
}

// Where the tiles of a map shorten: workgroups up to end[l] run tiles of
// cut_tile(l) pairs. A length is kept while two even shares of what is left,
// over the 1024 slots, are as long, so the workgroups end together and not
// with a last round of whole tiles (us, equal tiles / this: 600,000 pairs FP64
// 71 / 64, 3,000,017 mixed 191 / 181, 8,000,000 FP64 598 / 565 and mixed 439 /
// 419, 2^24 1171 / 1168). Tiles below 512 cost more in partly filled waves than
// they even out.
constexpr int CUT_LEVELS = 5;
struct TileCut {
    uint32_t end[CUT_LEVELS];
};

template <int TILE>
__host__ __device__ constexpr int cut_tile(int level) {
    constexpr int eighths[CUT_LEVELS] = {8, 6, 4, 3, 2};
    return TILE / 8 * eighths[level];
}

template <int TILE>
TileCut cut_tiles(int64_t n) {
    constexpr int64_t least = TILE < 512 ? TILE : 512, slots = 1024;
    TileCut c{};
    int64_t left = n, items = 0;
    for (int l = 0; l < CUT_LEVELS; l++) {
        const int64_t len = cut_tile<TILE>(l);
        const bool last = l + 1 == CUT_LEVELS || cut_tile<TILE>(l + 1) < least;
        const int64_t keep = last ? 0 : len * slots / 2;
        if (len >= least && left > keep) {
            const int64_t k = (left - keep + len - 1) / len;
            items += k;
            left -= k * len;
        }
        c.end[l] = uint32_t(items);
    }
    return c;
}

// Waves per SIMD the register allocation targets: the mixed form runs 2-3%
// faster at 5 (96 VGPRs, a few spills in its set-up code) than at the 4 its
// 125 VGPRs allow; the FP64 form is 1% slower at 5, so it keeps 4 (measured on
// 2^24 standard-rock pairs).
template <class P>
struct EvalWaves {
    static constexpr int value = 4;
};
template <>
struct EvalWaves<F32MN<1>> {
    static constexpr int value = 5;
};

// One workgroup per tile of up to TILE consecutive pairs.
template <class P, int TILE>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(EvalWaves<P>::value))) void dcs_eval_kernel(const double* __restrict__ K, const double* __restrict__ q,
                                                      int64_t n, DcsConsts c, Outs<typename P::out_t> o, TileCut cut) {
    __shared__ TileLists<TILE, P::has_redo> s;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];
    load_fm_tables(fm_block);  // published by run_tile's first barrier
    int64_t base = 0;
    uint32_t first = 0;  // of the level's workgroups
    int level = 0;
    for (; level + 1 < CUT_LEVELS && blockIdx.x >= cut.end[level]; level++) {
        base += int64_t(cut.end[level] - first) * cut_tile<TILE>(level);
        first = cut.end[level];
    }
    const int64_t len = cut_tile<TILE>(level);
    base += int64_t(blockIdx.x - first) * len;
    const int64_t end = (base + len < n) ? base + len : n;
    run_tile<P, TILE>(base, end, K, q, kernarg_consts(), o, s, fm::tab_from_block(fm_block));
}

// Maps that ask for closed forms only (bremsstrahlung, ionisation): one pair
// per thread and step, no tile, 44 registers and 8 waves per SIMD. Bound: HBM
// and VALU issue together. Measured on 2^24 pairs, FP64: bremsstrahlung 94 us
// (4.3 TB/s; 107 by the tile kernel), ionisation 74 (94), both 155 (167); mixed
// 57 (78), 59 (79), 83 (104).
inline int64_t closed_grid(int64_t n) {
    // four pairs per thread, up to 4096 workgroups, but at least one per CU
    // and SIMD slot while there are pairs: 2^20 pairs 8.7 us with 1024
    // workgroups, 10.1 with 4096; 2^24 94 with 4096, 99 with 1024
    return std::min<int64_t>(4096, std::max((n + 4 * WG - 1) / (4 * WG), std::min<int64_t>(1024, (n + WG - 1) / WG)));
}

template <class P>
__global__ __launch_bounds__(WG) void dcs_closed_kernel(const double* __restrict__ K, const double* __restrict__ q,
                                                        int64_t n, DcsConsts, Outs<typename P::out_t> o) {
    using out_t = typename P::out_t;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];
    const ConstsPtr cp = kernarg_consts();
    const int64_t stride = int64_t(gridDim.x) * WG;
    int64_t g = int64_t(blockIdx.x) * WG + threadIdx.x;
    double k = 1., qq = 0.;
    if (g < n) {
        k = K[g];
        qq = q[g];
    }
    load_fm_tables(fm_block);
    __syncthreads();
    const fm::Tab t = fm::tab_from_block(fm_block);
#pragma unroll 1
    while (g < n) {
        const DcsConsts& c = item_consts(cp);
        const int64_t next = g + stride;
        double k1 = 1., q1 = 0.;
        if (next < n) {
            k1 = K[next];
            q1 = q[next];
        }
        bool in = true;
        if constexpr (P::has_redo) in = P::in_range(k, qq, c);
        if (o.b) store_stream(&o.b[g], in ? P::brems(k, qq, c, t) : out_t(F64::brems(k, qq, c, t)));
        if (o.i) {
            if constexpr (P::has_redo)
                store_stream(&o.i[g], in ? P::ion(k, qq, c, t) : out_t(F64::ion_redo(k, qq, c, t)));
            else
                store_stream(&o.i[g], P::ion(k, qq, c, t));
        }
        g = next;
        k = k1;
        qq = q1;
    }
}

// run_tile reads c in place through kernarg_consts(), which locates it by
// TileKernelArgs: the kernel's leading parameters must stay (K, q, n, c).
static_assert(std::is_same<decltype(&dcs_eval_kernel<F64, 2048>),
                           void (*)(const double*, const double*, int64_t, DcsConsts, Outs<double>, TileCut)>::value,
              "dcs_eval_kernel's parameters must begin as TileKernelArgs lays them out");
static_assert(std::is_same<decltype(&dcs_small_kernel<double>),
                           void (*)(const double*, const double*, int64_t, DcsConsts, Outs<double>)>::value &&
                  std::is_same<decltype(&dcs_small_kernel<double>), decltype(&dcs_closed_kernel<F64>)>::value,
              "and dcs_small_kernel's and dcs_closed_kernel's with them");
static_assert(offsetof(TileKernelArgs, c) == 24, "three 8-byte arguments before the constants");

template <class P>
int launch_eval(const double* K, const double* q, int64_t n, const noa_dcs_element* el, double mass,
                Outs<typename P::out_t> o, hipStream_t stream) {
    if (int rc = check_element(el, mass)) return rc;
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0 (got %lld)", (long long)n);
    if (n == 0) return ok();
    if (!K || !q) return fail(NOA_DCS_EINVAL, "K and q must be non-NULL");
    if (!o.b && !o.p && !o.ph && !o.i) return ok();
    const int tile = eval_tile(n);
    if (n / tile > int64_t(0x7fffffff) - 4096) return fail(NOA_DCS_ERANGE, "n too large (%lld)", (long long)n);
    const DcsConsts c = make_consts(el->A, el->I, el->Z, mass);
    if (!o.p && !o.ph) {
        hipLaunchKernelGGL(dcs_closed_kernel<P>, dim3(uint32_t(closed_grid(n))), dim3(WG), 0, stream, K, q, n, c, o);
    } else if (tile == SMALL_TILE) {
        hipLaunchKernelGGL(dcs_small_kernel<typename P::out_t>, dim3(uint32_t((n + SMALL_TILE - 1) / SMALL_TILE)),
                           dim3(WG), 0, stream, K, q, n, c, o);
    } else {
        const TileCut cut = tile == 256 ? cut_tiles<256>(n) : tile == 1024 ? cut_tiles<1024>(n) : cut_tiles<2048>(n);
        auto* kernel = tile == 256    ? &dcs_eval_kernel<P, 256>
                       : tile == 1024 ? &dcs_eval_kernel<P, 1024>
                                      : &dcs_eval_kernel<P, 2048>;
        hipLaunchKernelGGL(kernel, dim3(cut.end[CUT_LEVELS - 1]), dim3(WG), 0, stream, K, q, n, c, o, cut);
    }
    if (int rc = check_hip(hipGetLastError(), "dcs_eval_kernel launch")) return rc;
    return ok();
}

// ---- seeded workload ----

__host__ __device__ inline uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__host__ __device__ inline double uniform53(uint64_t seed, uint64_t stream, uint64_t i) {
    const uint64_t key = mix64(seed * 0x9E3779B97F4A7C15ull + (stream + 1) * 0xD1B54A32D192ED03ull);
    const uint64_t z = mix64(key + (i + 1) * 0x9E3779B97F4A7C15ull);
    return double(z >> 11) * 0x1.0p-53;
}

__global__ __launch_bounds__(256) void fill_workload_kernel(double* __restrict__ K, double* __restrict__ q, int64_t n,
                                                            uint64_t seed, uint64_t s, double lk0, double lk1,
                                                            double ln0, double ln1) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
        const double u0 = uniform53(seed, 2 * s, uint64_t(i));
        const double u1 = uniform53(seed, 2 * s + 1, uint64_t(i));
        const double k = pow(10.0, lk0 + (lk1 - lk0) * u0);
        const double nu = pow(10.0, ln0 + (ln1 - ln0) * u1);
        K[i] = k;
        q[i] = nu * k;
    }
}

}  // namespace noa_hip

using namespace noa_hip;

extern "C" {

const char* noa_dcs_last_error(void) { return last_error_slot().c_str(); }

const char* noa_dcs_version(void) { return "noa_dcs 0.1.0 gfx950"; }

int noa_dcs_eval_f64(const double* K, const double* q, int64_t n, const noa_dcs_element* element, double mass,
                     const noa_dcs_outputs_f64* out, hipStream_t stream) {
    if (!out) return fail(NOA_DCS_EINVAL, "out is NULL");
    return launch_eval<F64>(K, q, n, element, mass, Outs<double>{out->brems, out->pair, out->photo, out->ion},
                            stream);
}

int noa_dcs_eval_f32mixed(const double* K, const double* q, int64_t n, const noa_dcs_element* element,
                          double mass, const noa_dcs_outputs_f32* out, hipStream_t stream) {
    if (!out) return fail(NOA_DCS_EINVAL, "out is NULL");
    return launch_eval<F32M>(K, q, n, element, mass, Outs<float>{out->brems, out->pair, out->photo, out->ion},
                             stream);
}

int noa_dcs_fill_workload(double* K, double* q, int64_t n, uint64_t seed, uint64_t stream_id, double lk0,
                          double lk1, double ln0, double ln1, hipStream_t stream) {
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0");
    if (n == 0) return ok();
    if (!K || !q) return fail(NOA_DCS_EINVAL, "K and q must be non-NULL");
    const int64_t blocks64 = (n + 255) / 256;
    const uint32_t blocks = uint32_t(blocks64 < 65536 ? blocks64 : 65536);
    hipLaunchKernelGGL(fill_workload_kernel, dim3(blocks), dim3(256), 0, stream, K, q, n, seed, stream_id, lk0, lk1,
                       ln0, ln1);
    if (int rc = check_hip(hipGetLastError(), "fill_workload_kernel launch")) return rc;
    return ok();
}

}  // extern "C"

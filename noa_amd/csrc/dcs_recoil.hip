// DEL / CEL recoil integrals of the four DCS processes over a vector of
// kinetic energies (src/noa/pms/dcs.hh:89-130, 444-497, 955-1001):
//   del_p(K) = (1/E) sum_j dcs_p(K, q_j) q_j   h w_j,   cel with q_j^2,
// i.e. (1/E) int dcs dq and (1/E) int dcs q dq over t = ln q, with
// q_j = exp(t_j) at the 6-node Gauss-Legendre points of ceil(min_points/6)
// subintervals of [ln(K xlow), ln K] (numerics.hh:72-108). Ionisation below
// K = (m - m_e)^2 / (2 m_e) takes the reference's analytic form.
//
// The DCS is the cost (180 evaluations per K and process at the reference's
// min_points = 180). One kernel does the whole of it: a workgroup takes a
// group of K values, evaluates their nodes like a map's tile (closed forms
// and exits per node, the open integrals compacted in LDS and drained by
// whole waves), keeps the node values in LDS and sums them there, so no
// (K, q) pair, no DCS value and no scratch goes through memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "capi_util.hh"
#include "dcs_consts.hh"
#include "dcs_f64.hh"
#include "dcs_tile.hh"
#include "fastmath.hh"
#include "launch_slices.hh"

namespace noa_hip {

// numerics.hh:97-100 (quadrature6 literals on [0, 1]).
static __constant__ double GL6_X[6] = {0.03376524, 0.16939531, 0.38069041, 0.61930959, 0.83060469, 0.96623476};
static __constant__ double GL6_W[6] = {0.08566225, 0.18038079, 0.23395697, 0.23395697, 0.18038079, 0.08566225};

constexpr int RECOIL_CHUNK = 65536;                            // K values the workspace is sized for
constexpr int64_t RECOIL_SCRATCH_BYTES = int64_t(32) << 20;  // as noa_dcs_recoil_noalloc_scratch_bytes reports

struct RecoilGrid {
    double xlow;
    int32_t n_itv;  // subintervals
    int32_t nodes;  // 6 n_itv
};

// dcs.hh:469-496 with the terms of :446-466.
__device__ __forceinline__ double analytic_ionisation(double K, double xlow, const DcsConsts& c, bool cel,
                                                      const fm::Tab& t) {
#pragma clang fp contract(off)
    const double me = ELECTRON_MASS;
    const double P2 = K * (K + c.i_2m);
    const double E = K + c.mass;
    const double Wmax = 2. * me * P2 / (c.i_m2 + me * (me + 2. * E));
    if (Wmax < X_FRACTION * K) return 0.;
    double Wmin = c.i_Wmin;
    const double qlow = K * xlow;
    if (qlow >= Wmin) Wmin = qlow;
    if (Wmax <= Wmin) return 0.;
    const double a0 = 0.5 / P2, a1 = -1. / Wmax, a2 = E * E / P2;
    double term;
    if (cel)
        term = 0.5 * a0 * (Wmax * Wmax - Wmin * Wmin) + a1 * (Wmax - Wmin) + a2 * fm::log(Wmax / Wmin, t);
    else
        term = a0 * (Wmax - Wmin) + a1 * fm::log(Wmax / Wmin, t) + a2 * (1. / Wmin - 1. / Wmax);
    return 1.535336E-05 * c.Zd / c.A * term;
}

// dcs.hh:955-1001: the ionisation integrals take the analytic form up to here.
__device__ __forceinline__ bool ion_is_analytic(double K, const DcsConsts& c) {
#pragma clang fp contract(off)
    const double m1 = c.mass - ELECTRON_MASS;
    return K <= 0.5 * m1 * m1 / ELECTRON_MASS;
}

// A workgroup's nodes in LDS, by item: node j of the group's K slot k at k nb + j.
template <int TILE>
struct RecoilLds {
    double q[TILE];
    double dcs[4][TILE];                // pair production: argmin until its integral has run
    double K[TILE / 6], lb[TILE / 6], h[TILE / 6];  // K, ln(K xlow) and the subinterval width, by K slot
    double part[TILE / 6][8];           // the DEL and CEL sums of a K
    double acc[8];                      // the sums of the node blocks before this one
    uint16_t photo_list[TILE], pair_list[TILE];
    uint32_t n_photo, n_pair;
};

// (SPLIT) the shared values and node terms of up to this many open integrals of
// either kind at a time.
constexpr int RECOIL_SPLIT = 192;
struct RecoilSplitLds {
    double x8[8], w8[8], x9[9], w9[9];
    double beta[RECOIL_SPLIT], tmin[RECOIL_SPLIT], a[8 * RECOIL_SPLIT], b[8 * RECOIL_SPLIT];
    F64::PhotoPre photo[RECOIL_SPLIT];
    double f[9 * RECOIL_SPLIT];
};
struct NoSplitLds {};

// Sum over the wave's lanes, in a fixed order, valid in lane 0.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Nodes per tile: two K values at min_points = 180, 360 nodes of 512 (lanes
// are 94% full whether a tile holds 1, 2 or 4 such K values). At 512 four
// workgroups fit a CU; tiles of 768 leave three and were as fast at 65,536 K
// and slower below, tiles of 256 (one K) 15% slower there.
constexpr int RECOIL_TILE = 512;

// One workgroup of LANES lanes per `group` K values; their nodes fit one tile, or (BLOCKS)
// group = 1 and the nodes go in blocks of TILE.
//
// Bound: FP64 VALU issue, as the map's tile kernel (the nodes have q >= K
// xlow, so nearly all open pair production and ~60% photonuclear: ~5000
// instructions each against the map's 2351). Passing the nodes through
// memory instead (a kernel that wrote (K, q) pairs, the map in tiles of 2048,
// and a sum per thread) took, at min_points 180, 444 us for 146 K values and
// 1790 us for 65,536, of which 296 and 320 us were the serial sums; this
// kernel takes 19 and 1567. At 30 points 189 -> 12 and 354 -> 336, at 6
// points 81 -> 15 and 167 -> 127.
// The nodes-in-blocks form is an instantiation of its own: its loop carries
// values that made the common one spill 28 registers.
template <int TILE, bool BLOCKS, int LANES, bool SPLIT = false>
__global__ __launch_bounds__(LANES) __attribute__((amdgpu_waves_per_eu(4))) void recoil_kernel(
    const double* __restrict__ K, int64_t n, DcsConsts, RecoilGrid g, int32_t group, Outs<double> del,
    Outs<double> cel) {
    __shared__ RecoilLds<TILE> s;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];
    __shared__ typename std::conditional<SPLIT, RecoilSplitLds, NoSplitLds>::type x;
    const ConstsPtr cp = vector_kernarg_consts();
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int i = tid; i < fm::TABLE_DOUBLES; i += LANES) fm_block[i] = fm::table_entry(i);
    if constexpr (SPLIT) {  // the node tables in LDS: the node index varies by lane
        if (tid < 9) {
            x.x9[tid] = GL9_X[tid];
            x.w9[tid] = GL9_W[tid];
            if (tid < 8) {
                x.x8[tid] = GL8_X[tid];
                x.w8[tid] = GL8_W[tid];
            }
        }
    }
    const fm::Tab t = fm::tab_from_block(fm_block);
    const bool want_b = del.b || cel.b, want_p = del.p || cel.p, want_ph = del.ph || cel.ph, want_i = del.i || cel.i;
    const int64_t k0 = int64_t(blockIdx.x) * group;
    const int nk = int(n - k0 < group ? n - k0 : group);
    __syncthreads();
    for (int kk = tid; kk < nk; kk += LANES) {
#pragma clang fp contract(off)
        const double k = K[k0 + kk];
        const double lb = fm::log(k * g.xlow, t);
        s.K[kk] = k;
        s.lb[kk] = lb;
        s.h[kk] = (fm::log(k, t) - lb) / double(uint32_t(g.n_itv));
    }
    for (int j0 = 0; j0 < (BLOCKS ? g.nodes : 1); j0 += TILE) {
        const int nb = BLOCKS && g.nodes - j0 > TILE ? TILE : g.nodes - j0;
        const int items = nk * nb;
        if (tid == 0) {
            s.n_photo = 0;
            s.n_pair = 0;
        }
        __syncthreads();
        // the nodes: closed forms, exits, the lists of open integrals
#pragma unroll 1
        for (int i0 = 0; i0 < items; i0 += LANES) {
            const DcsConsts& c = item_consts(cp);
            const int i = i0 + tid;
            bool pa = false, pha = false;
            if (i < items) {
                const int kk = i / nb;
                const int j = j0 + (i - kk * nb);
                const double k = s.K[kk];
                double q, am = 0.;
                {
#pragma clang fp contract(off)
                    q = fm::exp(s.lb[kk] + s.h[kk] * (double(uint32_t(j / 6)) + GL6_X[j % 6]), t);
                }
                s.q[i] = q;
                if (want_b) s.dcs[0][i] = F64::brems(k, q, c, t);
                if (want_i && !ion_is_analytic(k, c)) s.dcs[3][i] = F64::ion(k, q, c, t);
                if (want_p) {
                    pa = F64::pair_active(k, q, c, am);
                    s.dcs[1][i] = pa ? am : 0.;
                }
                if (want_ph) {
                    pha = F64::photo_active(k, q, c);
                    s.dcs[2][i] = 0.;
                }
            }
            if (want_ph) wave_append(pha, &s.n_photo, s.photo_list, uint32_t(i));
            if (want_p) wave_append(pa, &s.n_pair, s.pair_list, uint32_t(i));
        }
        __syncthreads();
        if constexpr (SPLIT) {
            // the integrals by quadrature node: a chain is a set-up, a node or
            // three and a sum, where an integral's own lane runs 8 or 9 in a row
            // (the sums are those of that loop, bit for bit)
            const uint32_t all_ph = s.n_photo, all_pa = s.n_pair;
#pragma unroll 1
            for (uint32_t e0 = 0; e0 < max(all_ph, all_pa); e0 += RECOIL_SPLIT) {
                const uint32_t nph = min(uint32_t(RECOIL_SPLIT), all_ph - min(e0, all_ph));
                const uint32_t npa = min(uint32_t(RECOIL_SPLIT), all_pa - min(e0, all_pa));
                const uint32_t pair0 = (nph + 63u) & ~63u, node0 = (9 * nph + 63u) & ~63u;
                const auto is_fast = [&](uint32_t i, const DcsConsts& c) {
                    return c.fast_ok && s.K[i / uint32_t(nb)] + c.mass <= F64::FAST_E_MAX;
                };
#pragma unroll 1
                for (uint32_t v = tid; v < pair0 + npa; v += LANES) {
                    const DcsConsts& c = item_consts(cp);
                    if (v < pair0) {
                        if (v >= nph) continue;
                        const uint32_t i = s.photo_list[e0 + v];
                        const double k = s.K[i / uint32_t(nb)];
                        if (is_fast(i, c))
                            x.photo[v] = F64::photo_setup<false, true>(k, s.q[i], c, t);
                        else
                            s.dcs[2][i] = F64::photo(k, s.q[i], c, t);
                    } else {
                        const uint32_t e = v - pair0, i = s.pair_list[e0 + e];
                        const double k = s.K[i / uint32_t(nb)];
                        if (is_fast(i, c)) {
                            double gamma;
                            const F64::PairPre p =
                                F64::pair_setup<false, true, true>(k, s.q[i], c, t, s.dcs[1][i], gamma);
                            x.beta[e] = p.beta;
                            x.tmin[e] = p.tmin;
                        } else {
                            s.dcs[1][i] = F64::pair_at(k, s.q[i], s.dcs[1][i], c, t);
                        }
                    }
                }
                __syncthreads();
#pragma unroll 1
                for (uint32_t v = tid; v < node0 + 8 * npa; v += LANES) {
                    const DcsConsts& c = item_consts(cp);
                    if (v < node0) {
                        if (v >= 9 * nph) continue;
                        const uint32_t e = v / 9, i = s.photo_list[e0 + e];
                        if (!is_fast(i, c)) continue;
                        const F64::PhotoPre p = x.photo[e];
                        x.f[v] = F64::photo_node<false, true>(p, x.x9[v - 9 * e], c, t);
                    } else {
                        const uint32_t u = v - node0, e = u / 8, j = u % 8, i = s.pair_list[e0 + e];
                        if (!is_fast(i, c)) continue;
                        const F64::PairPre p = F64::pair_pre(s.q[i], x.beta[e], x.tmin[e], c);
                        double a, b;
                        F64::pair_node<false, true>(p, x.x8[j], x.w8[j], c, t, a, b);
                        x.a[u] = a;
                        x.b[u] = b;
                    }
                }
                __syncthreads();
#pragma unroll 1
                for (uint32_t v = tid; v < pair0 + npa; v += LANES) {
                    const DcsConsts& c = item_consts(cp);
                    if (v < pair0) {
                        if (v >= nph) continue;
                        const uint32_t i = s.photo_list[e0 + v];
                        if (!is_fast(i, c)) continue;
                        double ds = 0.;
                        for (int j = 0; j < 9; j++) ds = F64::photo_add<false>(x.f[9 * v + j], x.w9[j], ds);
                        s.dcs[2][i] = F64::photo_finish<false, true>(s.K[i / uint32_t(nb)], x.photo[v], ds, c);
                    } else {
                        const uint32_t e = v - pair0, i = s.pair_list[e0 + e];
                        if (!is_fast(i, c)) continue;
                        double I = 0.;
                        for (int j = 0; j < 8; j++) I = F64::pair_add<false>(x.a[8 * e + j], x.b[8 * e + j], I);
                        const double k = s.K[i / uint32_t(nb)];
                        s.dcs[1][i] = F64::pair_finish<false, true>(k, s.q[i], F64::pair_gamma<true>(k, c), x.tmin[e],
                                                                    I, c, t);
                    }
                }
                __syncthreads();
            }
        } else {
            // the integrals, whole waves of one kind, photonuclear (heavier) first
            const uint32_t nph = s.n_photo;
            const uint32_t pair0 = (nph + 63u) & ~63u;
            const uint32_t total = pair0 + s.n_pair;
#pragma unroll 1
            for (uint32_t v = tid; v < total; v += LANES) {
                const DcsConsts& c = item_consts(cp);
                if (v < pair0) {
                    if (v >= nph) continue;
                    const uint32_t i = s.photo_list[v];
                    s.dcs[2][i] = F64::photo(s.K[i / uint32_t(nb)], s.q[i], c, t);
                } else {
                    const uint32_t i = s.pair_list[v - pair0];
                    s.dcs[1][i] = F64::pair_at(s.K[i / uint32_t(nb)], s.q[i], s.dcs[1][i], c, t);
                }
            }
        }
        __syncthreads();
        // sums: a wave takes one K
        for (int kk = wave; kk < nk; kk += LANES / 64) {
#pragma clang fp contract(off)
            double sum[8] = {};
            for (int l = lane; l < nb; l += 64) {
                const int i = kk * nb + l;
                const double q = s.q[i];
                const double hw = s.h[kk] * GL6_W[(j0 + l) % 6];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const double dq = s.dcs[p][i] * q;
                    sum[p] += dq * hw;
                    sum[4 + p] += dq * q * hw;
                }
            }
#pragma unroll
            for (int p = 0; p < 8; p++) sum[p] = wave_sum(sum[p]);
            if (lane == 0)
#pragma unroll
                for (int p = 0; p < 8; p++) s.part[kk][p] = sum[p];
        }
        __syncthreads();
        const bool last = !BLOCKS || j0 + TILE >= g.nodes;
        for (int v = tid; v < nk * 8; v += LANES) {
            const int kk = v / 8, p = v % 8;
            double acc = s.part[kk][p];
            if (BLOCKS && j0 > 0) acc += s.acc[p];  // (more than one node block: one K)
            if (!last) {
                s.acc[p] = acc;
            } else {
                const DcsConsts& c = item_consts(cp);
                const bool is_cel = p >= 4;
                const Outs<double>& out = is_cel ? cel : del;
                double* dst = (p & 3) == 0 ? out.b : (p & 3) == 1 ? out.p : (p & 3) == 2 ? out.ph : out.i;
                const double k = s.K[kk];
                double r = acc / (k + c.mass);
                if ((p & 3) == 3 && ion_is_analytic(k, c)) r = analytic_ionisation(k, g.xlow, c, is_cel, t);
                if (dst) dst[k0 + kk] = r;
            }
        }
    }
}

static_assert(std::is_same<decltype(&recoil_kernel<RECOIL_TILE, false, WG>),
                           void (*)(const double*, int64_t, DcsConsts, RecoilGrid, int32_t, Outs<double>,
                                    Outs<double>)>::value,
              "recoil_kernel's parameters must begin as VectorKernelArgs lays them out");

}  // namespace noa_hip

using namespace noa_hip;

namespace {

int64_t nodes_of(int32_t min_points) { return int64_t((uint32_t(min_points) + 5u) / 6u) * 6; }

int check_recoil_args(const double* K, int64_t n, double xlow, const noa_dcs_element* element, double mass,
                      int32_t min_points) {
    if (int rc = check_element(element, mass)) return rc;
    if (n < 0) return fail(NOA_DCS_EINVAL, "n must be >= 0");
    if (min_points < 1 || min_points > 6000) return fail(NOA_DCS_EINVAL, "min_points must be in [1, 6000]");
    if (!(xlow > 0.0 && xlow < 1.0)) return fail(NOA_DCS_EINVAL, "xlow must be in (0, 1) (got %g)", xlow);
    if (n > 0 && !K) return fail(NOA_DCS_EINVAL, "K is NULL");
    return NOA_DCS_OK;
}

// K values per workgroup: one as long as that fills the chip (1024 workgroups,
// 4 per CU), then as many as a tile holds; and at least a wave's worth of
// nodes. Measured (min_points 180, one / two K values per workgroup): 1000 K
// 43 / 51 us, 2000 K 77 / 76, 65,536 K 1802 / 1569; with 30 nodes each, 2000
// K 46 / 24.
int32_t recoil_group(int64_t n, int32_t nodes) {
    const int64_t want = std::max<int64_t>((n + 1023) / 1024, 64 / nodes);
    return int32_t(std::max<int64_t>(1, std::min<int64_t>(RECOIL_TILE / nodes, want)));
}

int recoil_run(const double* K, int64_t n, double xlow, const noa_dcs_element* element, double mass,
               int32_t min_points, const noa_dcs_outputs_f64& D, const noa_dcs_outputs_f64& C, hipStream_t stream) {
    const RecoilGrid g{xlow, int32_t((uint32_t(min_points) + 5u) / 6u), int32_t(nodes_of(min_points))};
    const DcsConsts c = make_consts(element->A, element->I, element->Z, mass);
    const int32_t group = recoil_group(n, g.nodes);
    const int64_t blocks = (n + group - 1) / group;
    const bool in_blocks = g.nodes > RECOIL_TILE;
    // up to 512 workgroups leave half of the chip's wave slots empty at 256
    // lanes each, and their length is the call's. Measured (us, 256 / 512 /
    // 1024 lanes; min_points 180): 146 K 27.9 / 20.3 / 20.4, 512 K 33.7 /
    // 28.3 / 37.7, 700 K 39.1 / 43.9 / 54.1; 1000 points, 146 K 96 / 67 / 60
    const bool wide = blocks <= 512;
    // up to one per CU also spread their integrals by node (1024 lanes): 6, 30
    // and 180 points 22.5 / 14.8, 20.0 / 12.4, 19.5 / 18.9 us for 146 K (a
    // CU's issue rate bounds the last)
    const bool by_node = blocks <= 256 && !in_blocks;
    const auto kernel = by_node ? &recoil_kernel<RECOIL_TILE, false, 4 * WG, true>
                        : wide  ? (in_blocks ? &recoil_kernel<RECOIL_TILE, true, 2 * WG>
                                             : &recoil_kernel<RECOIL_TILE, false, 2 * WG>)
                                : (in_blocks ? &recoil_kernel<RECOIL_TILE, true, WG>
                                             : &recoil_kernel<RECOIL_TILE, false, WG>);
    const int lanes = by_node ? 4 * WG : wide ? 2 * WG : WG;
    const int rc = launch_slices(blocks, lanes, [&](int64_t first, uint32_t count) {
        const int64_t k0 = first * group, nK = std::min<int64_t>(n - k0, int64_t(count) * group);
        auto shift = [k0](double* p) { return p ? p + k0 : nullptr; };
        const Outs<double> od{shift(D.brems), shift(D.pair), shift(D.photo), shift(D.ion)};
        const Outs<double> oc{shift(C.brems), shift(C.pair), shift(C.photo), shift(C.ion)};
        hipLaunchKernelGGL(kernel, dim3(count), dim3(lanes), 0, stream, K + k0, nK, c, g, group, od, oc);
        return check_hip(hipGetLastError(), "recoil_kernel");
    });
    if (rc) return rc;
    return ok();
}

}  // namespace

extern "C" {

int64_t noa_dcs_recoil_workspace_bytes(int64_t n, int32_t min_points) {
    if (n <= 0 || min_points < 1) return 0;
    return std::min<int64_t>(n, RECOIL_CHUNK) * nodes_of(min_points) * int64_t(6 * sizeof(double));
}

int noa_dcs_recoil_integrals_f64(const double* K, int64_t n, double xlow, const noa_dcs_element* element,
                                 double mass, int32_t min_points, const noa_dcs_outputs_f64* del,
                                 const noa_dcs_outputs_f64* cel, void* workspace, int64_t workspace_bytes,
                                 hipStream_t stream) {
    if (int rc = check_recoil_args(K, n, xlow, element, mass, min_points)) return rc;
    const noa_dcs_outputs_f64 none{nullptr, nullptr, nullptr, nullptr};
    const noa_dcs_outputs_f64& D = del ? *del : none;
    const noa_dcs_outputs_f64& C = cel ? *cel : none;
    if (n == 0 || !(D.brems || D.pair || D.photo || D.ion || C.brems || C.pair || C.photo || C.ion)) return ok();
    if (!workspace || workspace_bytes < noa_dcs_recoil_workspace_bytes(n, min_points))
        return fail(NOA_DCS_EINVAL, "workspace must hold noa_dcs_recoil_workspace_bytes(n, min_points) bytes");
    return recoil_run(K, n, xlow, element, mass, min_points, D, C, stream);
}

int64_t noa_dcs_recoil_noalloc_scratch_bytes(void) { return RECOIL_SCRATCH_BYTES; }

int noa_dcs_recoil_integrals_f64_noalloc(const double* K, int64_t n, double xlow, const noa_dcs_element* element,
                                         double mass, int32_t min_points, const noa_dcs_outputs_f64* del,
                                         const noa_dcs_outputs_f64* cel, hipStream_t stream) {
    if (int rc = check_recoil_args(K, n, xlow, element, mass, min_points)) return rc;
    const noa_dcs_outputs_f64 none{nullptr, nullptr, nullptr, nullptr};
    const noa_dcs_outputs_f64& D = del ? *del : none;
    const noa_dcs_outputs_f64& C = cel ? *cel : none;
    if (n == 0 || !(D.brems || D.pair || D.photo || D.ion || C.brems || C.pair || C.photo || C.ion)) return ok();
    return recoil_run(K, n, xlow, element, mass, min_points, D, C, stream);
}

}  // extern "C"

// Batched DCS evaluation over many elements with uneven pair counts, as one
// launch replayed from a hipGraph.
//
// The reference evaluates one element per adaptor call (src/noa/pms/dcs.hh:35-48);
// a material table of 48 elements with 2^10..2^20 pairs each would be 48
// launches, most of them far too small to fill 256 CUs. Here the pairs of all
// elements are cut into work items (element, begin, len <= TILE), ordered
// longest first, one workgroup each: the hardware hands the workgroups out in
// this order as slots come free, which is list scheduling. An item's element
// constants are read with scalar loads from a read-only table; the tile
// itself runs the same phased, compacting evaluation as the single-element
// kernel. Tile size and node-loop unroll are picked by timing the candidates
// on the actual batch, cached per (device, precision, shape).
//
// Measured on MI355X (us; a persistent grid that took equal items from an
// atomic counter, reset by a second kernel, against this), 48 elements of
// 2^10..2^20 pairs, 6.8e6 in all: FP64 545 / 508, mixed 429 / 365; 20 of
// 2^10..2^17, 4.1e5: 94 / 61, 93 / 55; 12 of 2^10..2^14, 6.6e4, in groups of
// 64 pairs: see SMALL_BATCH. The persistent loop held more constants across
// items than the SGPRs take (93 to 143 spills) and the mixed form could not
// run at the 5 waves per SIMD that it runs at here.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "capi_util.hh"
#include "dcs_consts.hh"
#include "dcs_f32m.hh"
#include "dcs_f64.hh"
#include "dcs_small.hh"
#include "dcs_tile.hh"
#include "launch_slices.hh"

namespace noa_hip {

struct WorkItem {
    int64_t begin;
    int32_t len;
    int32_t element;
};

// The item list and the element table are read-only for the whole launch:
// addressed through the constant address space their fields are scalar loads.
using ItemPtr = const __attribute__((address_space(4))) WorkItem*;

// Minimum resident waves per SIMD asked of the compiler, as for the
// single-element kernel. The unrolled FP64 form outgrows 256 VGPRs
// (1 wave/SIMD, spilling into the accumulator registers); bounded to 2 or 4
// it spills 1.1-1.6 KB per lane to scratch instead, so it stays unbounded.
template <class P, int TILE>
struct BatchMinWaves {
    static constexpr int value = std::is_same<P, F64N<2>>::value ? 1
                                 : TILE == 4096                  ? (P::has_redo ? 3 : 2)  // what the tile's LDS allows
                                 : std::is_same<P, F32MN<1>>::value ? 5
                                                                    : 4;
};

template <class P, int TILE>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(BatchMinWaves<P, TILE>::value))) void dcs_batch_kernel(
    const double* __restrict__ K, const double* __restrict__ q, const DcsConsts* __restrict__ consts,
    const WorkItem* __restrict__ items, Outs<typename P::out_t> o) {
    __shared__ TileLists<TILE, P::has_redo> s;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];
    load_fm_tables(fm_block);  // published by run_tile's first barrier
    const WorkItem& w = *(const WorkItem*)((ItemPtr)items + blockIdx.x);
    run_tile<P, TILE>(w.begin, w.begin + w.len, K, q, (ConstsPtr)(consts + w.element), o, s,
                      fm::tab_from_block(fm_block));
}

// Small batches: items of at most SMALL_TILE pairs, spread over lanes by
// quadrature node (dcs_small.hh).
template <class OutT>
__global__ __launch_bounds__(WG) void dcs_small_batch_kernel(const double* __restrict__ K,
                                                             const double* __restrict__ q,
                                                             const DcsConsts* __restrict__ consts,
                                                             const WorkItem* __restrict__ items, Outs<OutT> o) {
    __shared__ SmallLds s;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double fm_block[fm::TABLE_DOUBLES];
    const WorkItem& w = *(const WorkItem*)((ItemPtr)items + blockIdx.x);
    run_small<OutT>(w.begin, w.begin + w.len, K, q, (ConstsPtr)(consts + w.element), o, s, fm_block);
}

}  // namespace noa_hip

using namespace noa_hip;

struct noa_dcs_batch {
    int precision = 0;
    int tile = 0;
    int wpc = 0;             // workgroups resident per CU
    bool limit_wpc = false;  // at most wpc, as asked for; otherwise what registers and LDS allow
    int unroll = 1;
    bool small = false;  // items of SMALL_TILE pairs, dcs_small_batch_kernel
    const void* kernel = nullptr;
    size_t lds_pad = 0;
    int use_graph = 1;
    int n_cu = 0;
    int device = 0;
    double mass = 0;
    const double* K = nullptr;
    const double* q = nullptr;
    void* outs[4] = {nullptr, nullptr, nullptr, nullptr};
    std::vector<int64_t> offsets;
    std::vector<noa_dcs_element> elements;
    DcsConsts* d_consts = nullptr;
    WorkItem* d_items = nullptr;
    uint32_t n_items = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

std::mutex g_tune_mutex;

// A batch of up to this many pairs runs in items of 64, as maps of these
// sizes do (dcs_eval.hip, eval_tile): 6.6e4 pairs of 12 elements take 20 us, a
// replay's 5 included (32 in items of 512, 72 in tiles of 1024).
constexpr int64_t SMALL_BATCH = 200000;

template <class P>
const void* tile_kernel(int tile) {
    return tile == 1024   ? reinterpret_cast<const void*>(&dcs_batch_kernel<P, 1024>)
           : tile == 2048 ? reinterpret_cast<const void*>(&dcs_batch_kernel<P, 2048>)
                          : reinterpret_cast<const void*>(&dcs_batch_kernel<P, 4096>);
}

// The plan's kernel for its tile and unroll, and how many of its workgroups a
// CU holds. A limit asked for is kept by LDS that the kernel does not use.
int choose_kernel(noa_dcs_batch* b) {
    if (b->precision == NOA_DCS_PREC_F64)
        b->kernel = b->small         ? reinterpret_cast<const void*>(&dcs_small_batch_kernel<double>)
                    : b->unroll == 2 ? tile_kernel<F64N<2>>(b->tile)
                                     : tile_kernel<F64N<1>>(b->tile);
    else
        b->kernel = b->small         ? reinterpret_cast<const void*>(&dcs_small_batch_kernel<float>)
                    : b->unroll == 2 ? tile_kernel<F32MN<2>>(b->tile)
                                     : tile_kernel<F32MN<1>>(b->tile);
    b->lds_pad = 0;
    if (b->limit_wpc) {
        int per_block = 0, per_cu = 0;
        hipFuncAttributes attr;
        if (int rc = check_hip(hipFuncGetAttributes(&attr, b->kernel), "hipFuncGetAttributes")) return rc;
        if (int rc = check_hip(hipDeviceGetAttribute(&per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, b->device),
                               "hipDeviceGetAttribute"))
            return rc;
        if (int rc = check_hip(hipDeviceGetAttribute(
                                   &per_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, b->device),
                               "hipDeviceGetAttribute"))
            return rc;
        const int64_t want = std::min<int64_t>(per_block, per_cu / (b->wpc + 1) + 1024);
        b->lds_pad = size_t(std::max<int64_t>(0, want - int64_t(attr.sharedSizeBytes)));
        return NOA_DCS_OK;
    }
    if (int rc = check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b->wpc, b->kernel, WG, 0),
                           "hipOccupancyMaxActiveBlocksPerMultiprocessor"))
        return rc;
    b->wpc = std::max(1, b->wpc);
    return NOA_DCS_OK;
}

// (both output types: four pointers)
static_assert(sizeof(Outs<double>) == sizeof(Outs<float>) && sizeof(Outs<double>) == 4 * sizeof(void*),
              "noa_dcs_batch::outs stands for either");

hipError_t launch_direct(noa_dcs_batch* b, hipStream_t stream) {
    const int rc = launch_slices(b->n_items, WG, [&](int64_t first, uint32_t count) {
        const WorkItem* items = b->d_items + first;
        void* args[] = {&b->K, &b->q, &b->d_consts, &items, &b->outs};
        return int(hipLaunchKernel(b->kernel, dim3(count), dim3(WG), args, b->lds_pad, stream));
    });
    return hipError_t(rc);
}

// Work items, longest first. Tiles are `tile` pairs while much is left, then
// shorten with what is left, to two even shares of the 4 slots per CU and no
// less than `least`, so that the last ones end together. Measured (us;
// equal tiles against this): 4.1e5 pairs 69 / 61, 3.8e6 326 / 301, 1.2e7 903 /
// 895, mixed 636 / 618; `least` of 256 is slower from 4e5 pairs on, as the
// tiles of a map are (dcs_eval.hip, eval_tile).
std::vector<WorkItem> make_items(const noa_dcs_batch* b) {
    const std::vector<int64_t>& offsets = b->offsets;
    const int n_el = int(offsets.size()) - 1;
    int64_t left = offsets.back() - offsets.front();
    const int64_t least = left <= 300000 ? 256 : 512, slots = 4 * int64_t(b->n_cu);
    std::vector<int32_t> order(n_el);
    for (int e = 0; e < n_el; e++) order[e] = e;
    std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) {
        return offsets[x + 1] - offsets[x] > offsets[y + 1] - offsets[y];
    });
    std::vector<WorkItem> items;
    for (const int32_t e : order) {
        for (int64_t a = offsets[e]; a < offsets[e + 1];) {
            const int64_t share = (2 * left / slots + 63) / 64 * 64;
            const int64_t most = b->small ? SMALL_TILE : std::min<int64_t>(b->tile, std::max(least, share));
            const int64_t len = std::min(most, offsets[e + 1] - a);
            items.push_back(WorkItem{a, int32_t(len), e});
            a += len;
            left -= len;
        }
    }
    std::stable_sort(items.begin(), items.end(), [](const WorkItem& x, const WorkItem& y) { return x.len > y.len; });
    return items;
}

int upload_items(noa_dcs_batch* b) {
    if (int rc = choose_kernel(b)) return rc;
    const std::vector<WorkItem> items = make_items(b);
    if (items.size() > 0xffffffffull) return fail(NOA_DCS_ERANGE, "too many work items");
    if (b->d_items) (void)hipFree(b->d_items);
    b->d_items = nullptr;
    b->n_items = uint32_t(items.size());
    if (items.empty()) return NOA_DCS_OK;
    if (int rc = check_hip(hipMalloc(&b->d_items, items.size() * sizeof(WorkItem)), "hipMalloc(items)")) return rc;
    return check_hip(hipMemcpy(b->d_items, items.data(), items.size() * sizeof(WorkItem), hipMemcpyHostToDevice),
                     "hipMemcpy(items)");
}

// What a cache line is for. A batch that runs in small items has a line of its
// own: nothing of it is timed, and batches of the same size bucket on the
// other side of SMALL_BATCH must not take its values.
std::string tune_key(const noa_dcs_batch* b) {
    hipDeviceProp_t prop;
    (void)hipGetDeviceProperties(&prop, b->device);
    const int64_t total = b->offsets.back() - b->offsets.front();
    int lg = 0;
    while ((int64_t(1) << (lg + 1)) <= total) lg++;
    char buf[256];
    snprintf(buf, sizeof(buf), "%s|cu%d|prec%d|el%zu|log2n%d|%s|tile-wpc-unroll", prop.gcnArchName, b->n_cu,
             b->precision, b->elements.size(), lg, b->small ? "small-items" : "tiles");
    for (char* p = buf; *p; p++)
        if (*p == ' ') *p = '_';
    return buf;
}

// One line per configuration: key, tile, workgroups per CU (which the kernel
// decides; for the reader), unroll.
bool cache_lookup(const char* path, const std::string& key, int* tile, int* wpc, int* unroll) {
    if (!path) return false;
    FILE* f = fopen(path, "r");
    if (!f) return false;
    char line[512], k[256];
    int t, w, u;
    bool found = false;
    while (fgets(line, sizeof(line), f)) {
        if (sscanf(line, "%255s %d %d %d", k, &t, &w, &u) == 4 && key == k) {
            *tile = t;
            *wpc = w;
            *unroll = u;
            found = true;
        }
    }
    fclose(f);
    return found;
}

void cache_store(const char* path, const std::string& key, int tile, int wpc, int unroll) {
    if (!path) return;
    FILE* f = fopen(path, "a");
    if (!f) return;
    fprintf(f, "%s %d %d %d\n", key.c_str(), tile, wpc, unroll);
    fclose(f);
}

// Times the candidate tiles and node-loop unrolls, those that are not given, on
// the real batch and keeps the fastest. The outputs are overwritten with
// correct values by each run.
// Candidates are timed in turn, since the clock falls over the first
// milliseconds of load: one after the other, the first looked up to 6% faster
// than it was. Not among them, as never the fastest: tiles of 4096 (their LDS
// leaves 2 or 3 workgroups per CU: 6.8e6 pairs FP64 648 us against 492 in
// 2048) and the unrolled FP64 form (its registers leave one: 1111 us).
// A given tile leaves the mixed form's unroll to be timed: unrolled by two it
// is ahead where waves wait for each other and behind where the chip is full
// (us, unroll 1 / 2: 7.9e6 pairs in tiles of 2048 423 / 445, 5.9e5 70.8 / 70.0,
// 7.2e4 40.9 / 39.1).
int autotune(noa_dcs_batch* b, hipStream_t stream, bool tune_tile, bool tune_unroll) {
    std::vector<noa_dcs_batch> cand;
    for (const int t : {1024, 2048, 4096})
        for (const int u : {1, 2}) {
            if (tune_tile ? t == 4096 : t != b->tile) continue;
            if (tune_unroll ? u == 2 && b->precision == NOA_DCS_PREC_F64 : u != b->unroll) continue;
            cand.push_back(*b);
            cand.back().tile = t;
            cand.back().unroll = u;
        }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = check_hip(hipEventCreate(&e0), "hipEventCreate");
    if (!rc) rc = check_hip(hipEventCreate(&e1), "hipEventCreate");
    for (size_t k = 0; k < cand.size() && !rc; k++) rc = upload_items(&cand[k]);
    std::vector<float> best(cand.size(), 1e30f);
    for (int r = 0; r < 5 && !rc; r++) {  // (the first round warms up)
        for (size_t k = 0; k < cand.size() && !rc; k++) {
            (void)hipEventRecord(e0, stream);
            rc = check_hip(launch_direct(&cand[k], stream), "autotune launch");
            (void)hipEventRecord(e1, stream);
            if (!rc) rc = check_hip(hipEventSynchronize(e1), "autotune sync");
            float ms = 0;
            if (!rc) rc = check_hip(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
            if (r > 0) best[k] = std::min(best[k], ms);
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    const size_t win = size_t(std::min_element(best.begin(), best.end()) - best.begin());
    for (size_t k = 0; k < cand.size(); k++)
        if ((rc || k != win) && cand[k].d_items) (void)hipFree(cand[k].d_items);
    if (!rc) *b = cand[win];
    return rc;
}

int capture_graph(noa_dcs_batch* b, hipStream_t stream) {
    hipStream_t cs = stream;
    bool own = false;
    if (cs == nullptr) {  // the null stream cannot be captured
        if (int rc = check_hip(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking), "hipStreamCreate")) return rc;
        own = true;
    }
    int rc = check_hip(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    if (!rc) {
        const hipError_t le = launch_direct(b, cs);
        const hipError_t ee = hipStreamEndCapture(cs, &b->graph);
        rc = check_hip(le, "batch launch under capture");
        if (!rc) rc = check_hip(ee, "hipStreamEndCapture");
    }
    if (!rc) rc = check_hip(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0), "hipGraphInstantiate");
    if (own) (void)hipStreamDestroy(cs);
    return rc;
}

void release(noa_dcs_batch* b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    if (b->d_consts) (void)hipFree(b->d_consts);
    if (b->d_items) (void)hipFree(b->d_items);
    delete b;
}

}  // namespace

extern "C" {

int noa_dcs_batch_create(const noa_dcs_element* elements, const int64_t* offsets, int32_t n_elements, double mass,
                         const double* K, const double* q, void* out_brems, void* out_pair, void* out_photo,
                         void* out_ion, const noa_dcs_batch_config* config, hipStream_t stream,
                         noa_dcs_batch** plan) {
    if (!plan) return fail(NOA_DCS_EINVAL, "plan is NULL");
    *plan = nullptr;
    if (!elements || !offsets) return fail(NOA_DCS_EINVAL, "elements and offsets must be non-NULL");
    if (n_elements < 1) return fail(NOA_DCS_EINVAL, "n_elements must be >= 1");
    if (offsets[0] < 0) return fail(NOA_DCS_EINVAL, "offsets[0] must be >= 0");
    for (int e = 0; e < n_elements; e++) {
        if (offsets[e + 1] < offsets[e]) return fail(NOA_DCS_EINVAL, "offsets must be non-decreasing (element %d)", e);
        if (int rc = check_element(&elements[e], mass)) return rc;
    }
    if (!K || !q) return fail(NOA_DCS_EINVAL, "K and q must be non-NULL");
    const noa_dcs_batch_config def{NOA_DCS_PREC_F64, 0, 0, 1, nullptr, 0};
    const noa_dcs_batch_config& cfg = config ? *config : def;
    if (cfg.precision != NOA_DCS_PREC_F64 && cfg.precision != NOA_DCS_PREC_F32MIXED)
        return fail(NOA_DCS_EINVAL, "precision must be NOA_DCS_PREC_F64 or NOA_DCS_PREC_F32MIXED");
    if (cfg.tile != 0 && cfg.tile != 1024 && cfg.tile != 2048 && cfg.tile != 4096)
        return fail(NOA_DCS_EINVAL, "tile must be 0, 1024, 2048 or 4096 (got %d)", cfg.tile);
    if (cfg.waves_per_cu < 0 || cfg.waves_per_cu > 32)
        return fail(NOA_DCS_EINVAL, "waves_per_cu must be in [0, 32] (got %d)", cfg.waves_per_cu);
    if (cfg.unroll < 0 || cfg.unroll > 2)
        return fail(NOA_DCS_EINVAL, "unroll must be 0, 1 or 2 (got %d)", cfg.unroll);

    noa_dcs_batch* b = new noa_dcs_batch();
    b->precision = cfg.precision;
    b->use_graph = cfg.use_graph;
    b->mass = mass;
    b->K = K;
    b->q = q;
    b->outs[0] = out_brems;
    b->outs[1] = out_pair;
    b->outs[2] = out_photo;
    b->outs[3] = out_ion;
    b->offsets.assign(offsets, offsets + n_elements + 1);
    b->elements.assign(elements, elements + n_elements);
    int rc = check_hip(hipGetDevice(&b->device), "hipGetDevice");
    if (!rc) rc = check_hip(hipDeviceGetAttribute(&b->n_cu, hipDeviceAttributeMultiprocessorCount, b->device),
                            "hipDeviceGetAttribute");
    std::vector<DcsConsts> consts(n_elements);
    for (int e = 0; e < n_elements; e++) consts[e] = make_consts(elements[e].A, elements[e].I, elements[e].Z, mass);
    if (!rc) rc = check_hip(hipMalloc(&b->d_consts, consts.size() * sizeof(DcsConsts)), "hipMalloc(consts)");
    if (!rc)
        rc = check_hip(hipMemcpy(b->d_consts, consts.data(), consts.size() * sizeof(DcsConsts), hipMemcpyHostToDevice),
                       "hipMemcpy(consts)");
    if (!rc) {
        b->tile = cfg.tile ? cfg.tile : 2048;
        b->wpc = cfg.waves_per_cu;
        b->limit_wpc = cfg.waves_per_cu != 0;
        b->unroll = cfg.unroll ? cfg.unroll : 1;
        const bool all = cfg.tile == 0 && cfg.waves_per_cu == 0 && cfg.unroll == 0;
        b->small = all && offsets[n_elements] - offsets[0] <= SMALL_BATCH;
        const bool choice = cfg.tile == 0 || (cfg.unroll == 0 && cfg.precision == NOA_DCS_PREC_F32MIXED);
        if (!choice && !all) {  // nothing to time, to look up or to store: nothing to wait for
            rc = upload_items(b);
        } else {
            std::lock_guard<std::mutex> lock(g_tune_mutex);
            const std::string key = tune_key(b);
            int t = 0, w = 0, u = 0;
            const bool cached = all && cache_lookup(cfg.tune_cache, key, &t, &w, &u) &&
                                (t == 1024 || t == 2048 || t == 4096) && w >= 1 && w <= 32 && (u == 1 || u == 2);
            if (cached) {
                b->tile = t;
                b->unroll = u;
            }
            rc = cached || b->small ? upload_items(b) : autotune(b, stream, cfg.tile == 0, cfg.unroll == 0);
            if (!rc && all && !cached) cache_store(cfg.tune_cache, key, b->tile, b->wpc, b->unroll);
        }
    }
    if (!rc && b->use_graph && b->n_items) rc = capture_graph(b, stream);
    if (rc) {
        release(b);
        return rc;
    }
    *plan = b;
    return ok();
}

int noa_dcs_batch_launch(noa_dcs_batch* plan, hipStream_t stream) {
    if (!plan) return fail(NOA_DCS_EINVAL, "plan is NULL");
    if (plan->n_items == 0) return ok();
    if (plan->use_graph) {
        if (!plan->exec) return fail(NOA_DCS_ESTATE, "graph was not instantiated");
        if (int rc = check_hip(hipGraphLaunch(plan->exec, stream), "hipGraphLaunch")) return rc;
    } else {
        if (int rc = check_hip(launch_direct(plan, stream), "batch launch")) return rc;
    }
    return ok();
}

int noa_dcs_batch_info(const noa_dcs_batch* plan, int32_t* tile, int32_t* waves_per_cu, int32_t* unroll,
                       int64_t* n_items) {
    if (!plan) return fail(NOA_DCS_EINVAL, "plan is NULL");
    if (tile) *tile = plan->tile;
    if (waves_per_cu) *waves_per_cu = plan->wpc;
    if (unroll) *unroll = plan->unroll;
    if (n_items) *n_items = plan->n_items;
    return ok();
}

int noa_dcs_batch_destroy(noa_dcs_batch* plan) {
    if (!plan) return ok();
    release(plan);
    return ok();
}

}  // extern "C"

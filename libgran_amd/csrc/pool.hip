// Pools of independent DEM systems (include/hipgran.h, hg_pool_*): the
// batched and serving path.
//
// All systems of a pool live in one device arena of P particles (P = the
// pool's particle capacity); every per-particle array uses the same transposed
// layout as the single-system path with stride P, so a system is a contiguous
// index range [offset, offset + n) and a workgroup that owns it touches
// consecutive words.
//
// hg_pool_step launches one persistent kernel per rebuild interval. Each
// workgroup repeatedly takes the next system from a largest-first work queue
// and runs all steps of the interval for it: kick/drift of its own particles,
// workgroup barrier, acceleration pass (the same pair fold, walker and facet
// fold as the single-system kernels), barrier. A system's arithmetic does not
// depend on the other systems in the pool, so results are identical alone and
// in any mix. Between intervals a batched hashed cell list rebuilds the
// neighbour lists of the systems that are due, keyed by (system, cell).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <limits>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "pool_internal.h"
#include "snapshot.h"
#include "tile_step.h"

// Device scratch of hg_pool_energy_noalloc, the entry point that allocates
// nothing: the per-particle ledger terms of one system (8 doubles per
// particle) followed by their 8 sums, for systems of up to
// HG_NOALLOC_MAX_PARTICLES particles (8 MiB). Every GPU that runs the library
// holds its own copy until the process ends. Host code reaches it only through
// the address hipGetSymbolAddress returns for a device (noalloc_scratch),
// never through this name.
constexpr size_t kNoAllocParticles = HG_NOALLOC_MAX_PARTICLES;
static __device__ __align__(256) double scratch[8 * kNoAllocParticles + 8];

namespace hg {

namespace {

// Sums the per-particle ledger terms in particle order, the order sum_energy
// uses on the host: lane c < 7 adds term c of every particle, then lane 0 adds
// the seven sums; out[0..7].
__global__ void __launch_bounds__(64) k_energy_sum(const double *terms, uint32_t n, double *out) {
    __shared__ double part[7];
    const uint32_t c = threadIdx.x;
    if (c < 7) {
        double s = 0.0;
        for (uint32_t i = 0; i < n; i++) s += terms[8 * size_t(i) + c];
        part[c] = s;
    }
    __syncthreads();
    if (c < 7) out[c] = part[c];
    if (c == 0) {
        double t = 0.0;
        for (int q = 0; q < 7; q++) t += part[q];
        out[7] = t;
    }
}

// Zeroes `rows` strided rows [offset, offset+n) of an array with row stride.
__global__ void k_zero_rows_f64(double *p, size_t stride, size_t offset, size_t n, uint32_t rows) {
    const size_t total = rows * n;
    for (size_t k = blockIdx.x * size_t(blockDim.x) + threadIdx.x; k < total; k += size_t(gridDim.x) * blockDim.x)
        p[(k / n) * stride + offset + (k % n)] = 0.0;
}

inline unsigned nblk(size_t n, unsigned bs) { return unsigned((n + bs - 1) / bs); }

}  // namespace
hipError_t launch_tile_kick(const pool_view &V, const pool_view &Vo, const wide_block *map, unsigned blocks, int pairs,
                            double half, double dt, hipStream_t s) {
    if (blocks == 0) return hipSuccess;
    k_tile_kick<<<blocks, 64, 0, s>>>(V, Vo, map, uint32_t(tile_width(pairs)), half, dt);
    return hipGetLastError();
}
hipError_t launch_tile(const hg_params &p, const pool_view &Vi, const pool_view &Vo, const wide_block *map,
                              unsigned blocks, int mode, bool facets, double half, double dt, hipStream_t s) {
#define HG_TCASE(B, A)                                       \
    if (p.binary_model == B && p.pair_mode == A)             \
        return launch_tile_b<B, A>(p, Vi, Vo, map, blocks, mode, facets, half, dt, s);
    HG_TCASE(HG_BINARY_NONE, HG_PAIRS_ALL)
    HG_TCASE(HG_BINARY_NONE, HG_PAIRS_NEIGHBOR_LIST)
    HG_TCASE(HG_BINARY_CONTACT, HG_PAIRS_ALL)
    HG_TCASE(HG_BINARY_CONTACT, HG_PAIRS_NEIGHBOR_LIST)
    HG_TCASE(HG_BINARY_SINTER, HG_PAIRS_ALL)
    HG_TCASE(HG_BINARY_SINTER, HG_PAIRS_NEIGHBOR_LIST)
#undef HG_TCASE
    return hipErrorInvalidValue;
}
hipError_t launch_tile_steps(const hg_params &p, const pool_view &V, const pool_view &VB, const wide_block *map,
                                    unsigned blocks, uint32_t len, bool facets, double half, double dt,
                                    hipStream_t s) {
    const pool_view *in = len % 2 ? &VB : &V, *out = len % 2 ? &V : &VB;
    hipError_t e = launch_tile_kick(V, *in, map, blocks, p.pair_mode, half, dt, s);
    for (uint32_t k = 0; k < len && e == hipSuccess; k++) {
        e = launch_tile(p, *in, *out, map, blocks, k + 1 < len ? TILE_STEP : TILE_LAST, facets, half, dt, s);
        const pool_view *t = in;
        in = out;
        out = t;
    }
    return e;
}

namespace {

// The kicks of the walked systems (large all-pairs systems): before step s's
// pass the kick and drift (with `pending` = s > 0 the completion of step s - 1
// and the facets' move first), after the last pass its completion.
__global__ void __launch_bounds__(kWalkBlock) k_walk_kick(pool_view V, const wide_block *map, int pending, double half,
                                                          double dt) {
    const wide_block b = map[blockIdx.x];
    const pool_meta M = V.meta[b.slot];
    if (pending && b.start == 0 && threadIdx.x == 0)
        advance_facets(V.facets + size_t(b.slot) * V.max_facets, int(M.nf), dt);
    const uint32_t g = M.offset + b.start + threadIdx.x;
    if (g < M.offset + M.n) pool_kick_drift<STATE_GLOBAL>(V, M, pending != 0, half, dt, g, g + 1, 1);
}
__global__ void __launch_bounds__(kWalkBlock) k_walk_final(pool_view V, const wide_block *map, double half, double dt) {
    const wide_block b = map[blockIdx.x];
    const pool_meta M = V.meta[b.slot];
    if (b.start == 0 && threadIdx.x == 0) advance_facets(V.facets + size_t(b.slot) * V.max_facets, int(M.nf), dt);
    const uint32_t g = M.offset + b.start + threadIdx.x;
    if (g < M.offset + M.n) pool_final_kick<STATE_GLOBAL>(V, M, half, g, g + 1, 1);
}

hipError_t launch_walk(const hg_params &p, const pool_view &V, const wide_block *map, unsigned blocks, int pass,
                       hipStream_t s) {
    if (p.binary_model == HG_BINARY_NONE) return launch_walk_b<HG_BINARY_NONE>(p, V, map, blocks, pass, s);
    if (p.binary_model == HG_BINARY_CONTACT) return launch_walk_b<HG_BINARY_CONTACT>(p, V, map, blocks, pass, s);
    if (p.binary_model == HG_BINARY_SINTER) return launch_walk_b<HG_BINARY_SINTER>(p, V, map, blocks, pass, s);
    return hipErrorInvalidValue;
}
hipError_t launch_walk_steps(const hg_params &p, const pool_view &V, const wide_block *map, unsigned blocks,
                             uint32_t len, double half, double dt, hipStream_t s) {
    for (uint32_t k = 0; k < len; k++) {
        k_walk_kick<<<blocks, kWalkBlock, 0, s>>>(V, map, k > 0 ? 1 : 0, half, dt);
        const hipError_t e = launch_walk(p, V, map, blocks, int(k), s);
        if (e != hipSuccess) return e;
    }
    k_walk_final<<<blocks, kWalkBlock, 0, s>>>(V, map, half, dt);
    return hipGetLastError();
}

}  // namespace
}  // namespace hg

using namespace hg;

struct hg_pool {
    hg_params p{};
    int device = 0;  // the device current at hg_pool_create
    size_t P = 0, S = 0, MF = 0;
    // per-particle energy-ledger terms (hg_pool_energy), grown to the largest
    // system asked for
    double *energy = nullptr;
    size_t energy_cap = 0;
    hipStream_t stream = nullptr;
    double *x = nullptr, *v = nullptr, *th = nullptr, *w = nullptr, *a = nullptr, *al = nullptr;
    double *xb = nullptr, *vb = nullptr, *wb = nullptr;  // second x, v, omega for the per-step launches
    uint32_t cap_n = 0, *nb = nullptr, *ncnt = nullptr;
    uint32_t cap_s = 0, *pj[2] = {nullptr, nullptr}, *pcnt[2] = {nullptr, nullptr};
    uint32_t *bj = nullptr, *bcnt = nullptr;  // neck strengths (sinter_breaking)
    double *bstr = nullptr;
    double *ps[2] = {nullptr, nullptr};
    uint32_t *owner = nullptr;
    facet_dev *facets = nullptr, *facets_b = nullptr;  // facets_b: the second set of the per-step launches
    double *ss = nullptr;
    pool_meta *meta_d = nullptr;
    std::vector<pool_meta> meta;
    std::vector<uint64_t> step_index;
    std::vector<double> t;
    std::vector<char> active;
    std::vector<char> parked;  // out of the launch order while its state is read back
    std::vector<std::vector<std::pair<uint32_t, uint32_t>>> bonds;
    std::vector<size_t> skipped;
    uint32_t *order_d = nullptr, *counter_d = nullptr;
    std::vector<uint32_t> order;   // every active system, largest first
    uint32_t narrow_count = 0;     // systems below wide_min, uploaded to order_d
    uint32_t *packs_d = nullptr;   // the chunk kernel's queue: first | count << 24 over order_d
    uint32_t pack_count = 0;
    bool packing = true;           // small systems share a workgroup (neighbour-list mode)
    uint32_t wide_min = 0;         // systems with n >= wide_min use the wide launches (0: none)
    bool estimate = true;          // and others where split_order's estimate favours it
    uint32_t asked_min = 0;        // the two as the caller set them, which the tuner starts from
    bool asked_estimate = true;
    uint32_t wide_from = 0;        // the smallest system that does, in the order last used (0: none)
    wide_block *wide_map_d = nullptr;
    size_t wide_map_cap = 0;
    unsigned wide_blocks = 0;
    bool wide_walk = false;  // the wide systems are walked, not tiled (all pairs)
    // with wide systems present the wide launches run on stream_w beside the
    // chunk kernel, whose grid then leaves room worth wide_cus CUs
    hipStream_t stream_w = nullptr;
    hipStream_t stream_c = nullptr;  // copies that overlap an interval (pool_commit, pool_read_state)
    int n_cus = 0, wide_cus = 0;
    bool wide_graph = true;  // replay the wide launches of an interval as a HIP graph
    int tune_phase = 0;      // TUNE_*
    struct tune_cand {
        uint32_t wide_min;
        bool estimate;
        int wide_cus, tpb, wgs;  // launch split, chunk shape
    };
    std::vector<tune_cand> tune_cands;
    int tune_stage = 0;  // 0: chunk shapes, 1: launch splits
    std::vector<double> tune_scores;                   // seconds per step
    size_t tune_pos = 0;
    hipGraphExec_t wg_exec = nullptr;
    uint32_t wg_len = 0;
    bool wg_facets = false, wg_walk = false;
    unsigned wg_blocks = 0;
    double wg_dt = 0.0;
    hipEvent_t wev[3] = {nullptr, nullptr, nullptr};
    double last_wide_ms = 0.0;
    uint64_t last_wide_launches = 0;
    bool order_dirty = true;
    bool meta_dirty = true;
    uint32_t hash_size = 0, *cell_of = nullptr, *buckets = nullptr, *bucket_start = nullptr, *scan_tmp = nullptr;
    cell_rec *cell_recs = nullptr;
    int *flags = nullptr, *flags_host = nullptr;
    host_stage stage;
    // per-system fault words set by the kernels (device, cleared after every
    // read) and the faults recorded so far (host, per slot)
    int *sflags = nullptr, *sflags_host = nullptr;
    std::vector<int> fault;
    int fault_nl_need = 0, fault_pair_need = 0;  // counts the last overflows needed
    std::map<uint32_t, uint32_t> free_ranges;  // offset -> length
    uint32_t high_water = 0;
    std::vector<void *> allocations;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    hipEvent_t evb[2] = {nullptr, nullptr};  // start and end of an interval's device work
    pool_meta *meta_pinned = nullptr;        // staging of the per-interval meta upload
    double last_busy_ms = 0.0;
    // the interval queued by pool_begin and not yet closed by pool_end
    struct {
        bool active = false;
        uint32_t len = 0, count = 0;
        bool rebuilt = false, wide = false;
        double dt = 0.0;
        std::chrono::steady_clock::time_point t0;
    } fl;
    double last_chunk_ms = 0.0, last_rebuild_ms = 0.0;
    uint64_t last_chunks = 0, last_chunk_steps = 0;
    int grid = 0;
    uint32_t lds_cap = 0;
    size_t lds_bytes_per_wg = 0;
    size_t lds_per_cu = 0, lds_per_block = 0;  // device limits
    int wg_per_cu = 2;                         // chunk-kernel workgroups per CU
    int chunk_tpb = 256;                       // and their threads
};

namespace {

template <typename T>
hg_status palloc(hg_pool *Q, T **p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc(reinterpret_cast<void **>(p), count * sizeof(T));
    if (e != hipSuccess)
        return fail(e == hipErrorOutOfMemory ? HG_ERR_OOM : HG_ERR_HIP,
                    "pool: hipMalloc of " + std::to_string(count * sizeof(T)) + " bytes: " + hipGetErrorString(e));
    Q->allocations.push_back(*p);
    return HG_OK;
}

#define PG_TRY(expr)                  \
    do {                              \
        hg_status st_ = (expr);       \
        if (st_ != HG_OK) return st_; \
    } while (0)

uint32_t pool_cap_n(const hg_params &p) {
    if (p.pair_mode != HG_PAIRS_NEIGHBOR_LIST) return 0;
    if (p.neighbor_capacity) return p.neighbor_capacity;
    const double r = p.contact.r_part > 0 ? p.contact.r_part : (p.sinter.r_part > 0 ? p.sinter.r_part : p.hamaker.r_part);
    double ratio = r > 0 ? p.r_verlet / r : 64.0;
    double bound = 0.7405 * (std::pow(ratio + 1.0, 3.0) - 1.0) * 1.3;
    return uint32_t(std::ceil(std::max(bound, 8.0) / 8.0) * 8.0);
}

uint32_t pool_cap_s(const hg_params &p) {
    if (p.binary_model == HG_BINARY_NONE) return 0;
    return std::max<uint32_t>(p.pair_capacity ? p.pair_capacity : 24u, kTagPrefetch);
}

// Looks at the flag words that pool_begin copied back after its launches (the
// stream has been waited for). When one is raised, the
// per-system fault words say which systems tripped it: they are added to
// Q->fault (those systems are no longer stepped) and pushed onto `faulted`,
// and both the flags and the fault words are cleared on the device.
hg_status collect_faults(hg_pool *Q, std::vector<int32_t> &faulted) {
    const int *f = Q->flags_host;
    if (!f[FLAG_NL_OVERFLOW] && !f[FLAG_PAIR_OVERFLOW] && !f[FLAG_NUMERIC]) return HG_OK;
    if (f[FLAG_NL_OVERFLOW]) Q->fault_nl_need = std::max(Q->fault_nl_need, f[FLAG_NL_MAXCOUNT]);
    if (f[FLAG_PAIR_OVERFLOW]) Q->fault_pair_need = std::max(Q->fault_pair_need, f[FLAG_PAIR_MAXCOUNT]);
    HG_HIP(hipMemcpyAsync(Q->sflags_host, Q->sflags, Q->S * sizeof(int), hipMemcpyDeviceToHost, Q->stream));
    HG_HIP(hipStreamSynchronize(Q->stream));
    for (size_t s = 0; s < Q->S; s++) {
        if (!Q->sflags_host[s] || !Q->active[s]) continue;
        if (!Q->fault[s]) faulted.push_back(int32_t(s));
        Q->fault[s] |= Q->sflags_host[s];
        Q->order_dirty = true;
    }
    HG_HIP(launch_zero_u32(reinterpret_cast<uint32_t *>(Q->flags), FLAG_COUNT, Q->stream));
    HG_HIP(launch_zero_u32(reinterpret_cast<uint32_t *>(Q->sflags), Q->S, Q->stream));
    HG_HIP(hipStreamSynchronize(Q->stream));
    return HG_OK;
}

// k chunk-kernel workgroups per CU (the grid), each with 1/k of the CU's
// LDS (less the static words) for its system's state and partner ids.
void set_chunk_wgs(hg_pool *Q, int k) {
    Q->wg_per_cu = k;
    Q->grid = Q->n_cus * k;
    size_t per_wg = std::min<size_t>(Q->lds_per_block, Q->lds_per_cu / size_t(k));
    per_wg = per_wg > 1024 ? per_wg - 1024 : 0;
    Q->lds_cap = uint32_t(per_wg);
    Q->lds_bytes_per_wg = per_wg;
}

pool_view make_pool_view(hg_pool *Q) {
    pool_view V;
    V.x = Q->x; V.v = Q->v; V.th = Q->th; V.w = Q->w; V.a = Q->a; V.al = Q->al;
    V.nb = Q->nb;
    V.ncnt = Q->ncnt;
    V.pj0 = Q->pj[0]; V.pj1 = Q->pj[1];
    V.pcnt0 = Q->pcnt[0]; V.pcnt1 = Q->pcnt[1];
    V.ps0 = Q->ps[0]; V.ps1 = Q->ps[1];
    V.cap_s = Q->cap_s;
    V.bj = Q->bj;
    V.bstr = Q->bstr;
    V.bcnt = Q->bcnt;
    V.cap_n = Q->cap_n;
    V.facets = Q->facets;
    V.max_facets = uint32_t(Q->MF);
    V.facet_steps = 1;
    V.ss = Q->ss;
    V.meta = Q->meta_d;
    V.stride = Q->P;
    V.flags = Q->flags;
    V.sflags = Q->sflags;
    return V;
}

hg_status valid_slot(hg_pool *Q, int32_t slot) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (slot < 0 || size_t(slot) >= Q->S || !Q->active[slot]) return fail(HG_ERR_INVALID, "no such system in the pool");
    return HG_OK;
}

hg_status upload_meta(hg_pool *Q) {
    HG_HIP(hipMemcpyAsync(Q->meta_d, Q->meta.data(), Q->S * sizeof(pool_meta), hipMemcpyHostToDevice, Q->stream));
    HG_HIP(hipStreamSynchronize(Q->stream));
    Q->meta_dirty = false;
    return HG_OK;
}

// Copies strided rows [offset, offset+n) of a device array into a host array
// with row stride n; `width` elements per particle (a row of the device array
// holds P*width elements).
template <typename T>
hg_status download_rows(hg_pool *Q, const T *dev, uint32_t offset, uint32_t n, uint32_t rows, T *host,
                        size_t width = 1) {
    if (rows == 0 || n == 0) return HG_OK;
    const size_t row = n * width * sizeof(T);
    HG_HIP(hipMemcpy2DAsync(host, row, dev + offset * width, Q->P * width * sizeof(T), row, rows,
                            hipMemcpyDeviceToHost, Q->stream));
    HG_HIP(hipStreamSynchronize(Q->stream));
    return HG_OK;
}

hg_status rebuild_due(hg_pool *Q) {
    const uint32_t hw = Q->high_water;
    if (hw == 0) return HG_OK;
    const list_build B{Q->x,         hw,          Q->P,       Q->p.r_verlet, Q->owner, Q->meta_d, Q->hash_size, Q->buckets,
                       Q->bucket_start, Q->scan_tmp, Q->cell_of, Q->cell_recs,  Q->nb,    Q->ncnt,   Q->cap_n,     Q->flags,
                       Q->sflags};
    HG_HIP(launch_cell_lists(B, Q->stream));
    return HG_OK;
}

// Inputs of the energy ledger of one system of the pool.
energy_view pool_energy_view(hg_pool *Q, const pool_meta &M) {
    const bool nl = Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST, tab = Q->cap_s != 0;
    return energy_view{Q->x,
                       Q->v,
                       Q->w,
                       M.offset,
                       M.n,
                       Q->P,
                       nl ? Q->nb : nullptr,
                       nl ? Q->ncnt : nullptr,
                       tab ? Q->pj[M.cur] : nullptr,
                       tab ? Q->pcnt[M.cur] : nullptr,
                       tab ? Q->ps[M.cur] : nullptr,
                       nullptr,
                       nullptr,
                       nullptr,
                       nullptr};
}

// The device address of `scratch` on device dev: looked up once per device,
// with that device current, the first time a call reaches it; later calls
// reuse it.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch[kMaxDevices] = {};

hg_status noalloc_scratch(int dev, double **out) {
    if (dev < 0 || dev >= kMaxDevices) return fail(HG_ERR_INVALID, "device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev]) {
        int cur = 0;
        HG_HIP(hipGetDevice(&cur));
        if (cur != dev) HG_HIP(hipSetDevice(dev));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != dev) (void)hipSetDevice(cur);
        HG_HIP(e);
        g_scratch[dev] = static_cast<double *>(p);
    }
    *out = g_scratch[dev];
    return HG_OK;
}

}  // namespace

extern "C" {

size_t hg_pool_bytes_per_particle(const hg_params *p, size_t max_facets) {
    if (!p) return 0;
    const size_t cap_n = pool_cap_n(*p), cap_s = pool_cap_s(*p);
    size_t b = 9 * 32;                   // x, v, theta, omega, a, alpha; second x, v, omega
    b += cap_n * 4 + 4;                  // neighbour slots + count
    b += 2 * (cap_s * (4 + 8 * kSpringRec) + 4);  // pair-state table, double buffered
    b += max_facets * 72;                // facet springs
    b += 4;                              // owner
    if (p->binary_model == HG_BINARY_SINTER && p->sinter_breaking)
        b += kMaxBondsPerParticle * 12 + 4;  // neck-strength lists
    if (p->pair_mode == HG_PAIRS_NEIGHBOR_LIST) b += 4 + 32 + 3 * 2 * 4 + 4;  // cell list scratch
    else b += sizeof(wide_block);  // tiles of one particle
    return b;
}

hg_status hg_pool_create(const hg_params *params, size_t max_particles, size_t max_systems, size_t max_facets,
                         hg_pool **out) {
    if (!out || !params) return fail(HG_ERR_INVALID, "hg_pool_create: params and out are required");
    *out = nullptr;
    if (max_particles == 0 || max_particles >= (size_t(1) << 31) || max_systems == 0 ||
        max_systems >= (size_t(1) << 24))
        return fail(HG_ERR_INVALID, "hg_pool_create: need 0 < max_particles < 2^31 and 0 < max_systems < 2^24");
    if (max_facets > size_t(kMaxFacets)) return fail(HG_ERR_INVALID, "hg_pool_create: at most 16 facets per system");
    if (params->precision != HG_PRECISION_FP64 && params->precision != HG_PRECISION_MIXED)
        return fail(HG_ERR_INVALID, "hg_pool_create: unknown precision");
    if (params->binary_model < HG_BINARY_NONE || params->binary_model > HG_BINARY_SINTER)
        return fail(HG_ERR_INVALID, "hg_pool_create: pools run no binary functor, contact_force, alt_sinter or "
                                    "alt_breaking_sinter; the legacy sinter_functor runs on single systems");
    if (params->hamaker_model < HG_HAMAKER_NONE || params->hamaker_model > HG_HAMAKER_SIMPLIFIED)
        return fail(HG_ERR_INVALID, "hg_pool_create: unknown hamaker_model");
    if (params->sinter_breaking != 0 && (params->sinter_breaking != 1 || params->binary_model != HG_BINARY_SINTER))
        return fail(HG_ERR_INVALID, "hg_pool_create: sinter_breaking is 0, or 1 with HG_BINARY_SINTER");
    if (params->pair_mode == HG_PAIRS_NEIGHBOR_LIST && !(params->r_verlet > 0.0))
        return fail(HG_ERR_INVALID, "hg_pool_create: neighbour-list mode needs r_verlet > 0");
    if (params->facet_advance != 0)
        return fail(HG_ERR_INVALID, "hg_pool_create: pools advance facets after every step (facet_advance = 0)");
    int dev = 0;
    HG_HIP(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    HG_HIP(hipGetDeviceProperties(&prop, dev));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(HG_ERR_NO_DEVICE, std::string("hipgran is built for gfx950; current device is ") + prop.gcnArchName);

    hg_pool *Q = new hg_pool();
    auto bail = [&](hg_status st) {
        std::string msg = hg_last_error();
        hg_pool_destroy(Q);
        fail(st, msg);
        return st;
    };
#define PG_TRYC(expr)                           \
    do {                                        \
        hg_status st_ = (expr);                 \
        if (st_ != HG_OK) return bail(st_);     \
    } while (0)
#define PG_HIPC(call)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess)                                                                  \
            return bail(fail(HG_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_))); \
    } while (0)
    Q->p = *params;
    Q->device = dev;
    Q->P = max_particles;
    Q->S = max_systems;
    Q->MF = max_facets;
    Q->n_cus = prop.multiProcessorCount;
    Q->lds_per_cu = prop.maxSharedMemoryPerMultiProcessor;
    Q->lds_per_block = prop.sharedMemPerBlock;
    set_chunk_wgs(Q, 2);
    PG_HIPC(hipStreamCreateWithFlags(&Q->stream, hipStreamNonBlocking));
    for (auto &e : Q->ev) PG_HIPC(hipEventCreate(&e));
    for (auto &e : Q->wev) PG_HIPC(hipEventCreate(&e));
    for (auto &e : Q->evb) PG_HIPC(hipEventCreate(&e));
    Q->wide_min = Q->asked_min = kDefaultWideMin;
    Q->wide_cus = int(std::lround(kDefaultWideCuFraction * Q->n_cus));
    PG_HIPC(hipStreamCreateWithFlags(&Q->stream_w, hipStreamNonBlocking));
    PG_HIPC(hipStreamCreateWithFlags(&Q->stream_c, hipStreamNonBlocking));
    const size_t P = Q->P;
    double **fields[9] = {&Q->x, &Q->v, &Q->th, &Q->w, &Q->a, &Q->al, &Q->xb, &Q->vb, &Q->wb};
    for (auto f : fields) PG_TRYC(palloc(Q, f, 4 * P));
    Q->cap_n = pool_cap_n(Q->p);
    Q->cap_s = pool_cap_s(Q->p);
    if (Q->cap_n) {
        PG_TRYC(palloc(Q, &Q->nb, size_t(Q->cap_n) * P));
        PG_TRYC(palloc(Q, &Q->ncnt, P));
        PG_HIPC(launch_zero_u32(Q->ncnt, P, Q->stream));
        uint32_t hs = 1024;
        while (hs < 2 * P && hs < (1u << 30)) hs <<= 1;
        Q->hash_size = hs;
        PG_TRYC(palloc(Q, &Q->cell_of, P));
        PG_TRYC(palloc(Q, &Q->cell_recs, P));
        PG_TRYC(palloc(Q, &Q->buckets, size_t(2) * hs));
        PG_TRYC(palloc(Q, &Q->bucket_start, hs));
        PG_TRYC(palloc(Q, &Q->scan_tmp, scan_tmp_words(hs)));
    }
    if (Q->cap_s) {
        for (int b = 0; b < 2; b++) {
            PG_TRYC(palloc(Q, &Q->pj[b], size_t(Q->cap_s) * P));
            PG_TRYC(palloc(Q, &Q->ps[b], size_t(Q->cap_s) * kSpringRec * P));
            PG_TRYC(palloc(Q, &Q->pcnt[b], P));
        }
    }
    if (Q->p.binary_model == HG_BINARY_SINTER && Q->p.sinter_breaking) {
        PG_TRYC(palloc(Q, &Q->bj, size_t(kMaxBondsPerParticle) * P));
        PG_TRYC(palloc(Q, &Q->bstr, size_t(kMaxBondsPerParticle) * P));
        PG_TRYC(palloc(Q, &Q->bcnt, P));
        PG_HIPC(launch_zero_u32(Q->bcnt, P, Q->stream));
    }
    PG_TRYC(palloc(Q, &Q->owner, P));
    {
        std::vector<uint32_t> none(P, kNoEntry);
        // not hipMemcpy: the default stream refuses it, and spoils the recording,
        // while another thread's pool records a graph
        PG_HIPC(hipMemcpyAsync(Q->owner, none.data(), P * 4, hipMemcpyHostToDevice, Q->stream));
        PG_HIPC(hipStreamSynchronize(Q->stream));
    }
    PG_TRYC(palloc(Q, &Q->facets, std::max<size_t>(1, Q->S * std::max<size_t>(Q->MF, 1))));
    PG_TRYC(palloc(Q, &Q->facets_b, std::max<size_t>(1, Q->S * std::max<size_t>(Q->MF, 1))));
    if (Q->MF) PG_TRYC(palloc(Q, &Q->ss, Q->MF * 9 * P));
    PG_TRYC(palloc(Q, &Q->meta_d, Q->S));
    PG_TRYC(palloc(Q, &Q->order_d, Q->S));
    PG_TRYC(palloc(Q, &Q->packs_d, Q->S));
    Q->wide_map_cap = Q->P / size_t(tile_width(Q->p.pair_mode)) + Q->S + 1;
    PG_TRYC(palloc(Q, &Q->wide_map_d, Q->wide_map_cap));
    PG_TRYC(palloc(Q, &Q->counter_d, 1));
    PG_TRYC(palloc(Q, &Q->flags, FLAG_COUNT));
    PG_TRYC(palloc(Q, &Q->sflags, Q->S));
    PG_HIPC(hipHostMalloc(reinterpret_cast<void **>(&Q->flags_host), FLAG_COUNT * sizeof(int)));
    PG_HIPC(hipHostMalloc(reinterpret_cast<void **>(&Q->sflags_host), Q->S * sizeof(int)));
    PG_HIPC(hipHostMalloc(reinterpret_cast<void **>(&Q->meta_pinned), Q->S * sizeof(pool_meta)));
    PG_HIPC(launch_zero_u32(reinterpret_cast<uint32_t *>(Q->flags), FLAG_COUNT, Q->stream));
    PG_HIPC(launch_zero_u32(reinterpret_cast<uint32_t *>(Q->sflags), Q->S, Q->stream));
    Q->meta.assign(Q->S, pool_meta{0, 0, 0, 0, 0, 0, 0, 0});
    Q->step_index.assign(Q->S, 0);
    Q->t.assign(Q->S, 0.0);
    Q->active.assign(Q->S, 0);
    Q->parked.assign(Q->S, 0);
    Q->fault.assign(Q->S, 0);
    Q->bonds.assign(Q->S, {});
    Q->skipped.assign(Q->S, 0);
    Q->free_ranges[0] = uint32_t(P);
    PG_TRYC(upload_meta(Q));
    *out = Q;
    return HG_OK;
#undef PG_TRYC
#undef PG_HIPC
}

hg_status hg_pool_destroy(hg_pool *Q) {
    if (!Q) return HG_OK;
    if (Q->stream) (void)hipStreamSynchronize(Q->stream);
    if (Q->stream_w) (void)hipStreamSynchronize(Q->stream_w);
    if (Q->stream_c) (void)hipStreamSynchronize(Q->stream_c);
    for (void *p : Q->allocations) (void)hipFree(p);
    for (auto e : Q->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto e : Q->wev)
        if (e) (void)hipEventDestroy(e);
    for (auto e : Q->evb)
        if (e) (void)hipEventDestroy(e);
    if (Q->meta_pinned) (void)hipHostFree(Q->meta_pinned);
    if (Q->wg_exec) (void)hipGraphExecDestroy(Q->wg_exec);
    if (Q->stream_w) (void)hipStreamDestroy(Q->stream_w);
    if (Q->stream_c) (void)hipStreamDestroy(Q->stream_c);
    if (Q->flags_host) (void)hipHostFree(Q->flags_host);
    if (Q->sflags_host) (void)hipHostFree(Q->sflags_host);
    if (Q->stream) (void)hipStreamDestroy(Q->stream);
    delete Q;
    return HG_OK;
}

}  // extern "C"

namespace hg {

hg_status pool_prepare(const hg_params &p, size_t n, const double *x0, const double *v0, const double *theta0,
                       const double *omega0, const std::vector<std::pair<uint32_t, uint32_t>> *given_bonds,
                       size_t given_skipped, pool_prep &out) {
    if (!x0) return fail(HG_ERR_INVALID, "hg_pool_add: x0 is required");
    if (n == 0) return fail(HG_ERR_INVALID, "hg_pool_add: empty system");
    out.n = n;
    out.bonds.clear();
    out.skipped = 0;
    out.rows.assign(p.binary_model == HG_BINARY_SINTER ? n : 0, {});
    if (p.binary_model == HG_BINARY_SINTER) {
        if (given_bonds) {
            out.bonds = *given_bonds;
            out.skipped = given_skipped;
        } else {
            sinter_topology_host(n, x0, p.sinter.r_part, p.sinter.d_crit, out.bonds, out.skipped, !p.sinter_breaking);
        }
        for (auto &b : out.bonds) {
            out.rows[b.first].push_back(b.second | kBondBit);
            out.rows[b.second].push_back(b.first | kBondBit);
        }
        for (auto &r : out.rows)
            std::sort(r.begin(), r.end(), [](uint32_t a, uint32_t b) { return (a & kIdxMask) < (b & kIdxMask); });
    }
    const double *src[4] = {x0, v0, theta0, omega0};
    for (int f = 0; f < 4; f++) {
        out.q4[f].assign(4 * n, 0.0);
        if (src[f])
            for (size_t i = 0; i < n; i++)
                for (int c = 0; c < 3; c++) out.q4[f][4 * i + c] = src[f][3 * i + c];
    }
    return HG_OK;
}

hg_status pool_commit(hg_pool *Q, pool_prep &prep, int32_t *slot_out, hipStream_t cs) {
    if (!cs && Q) cs = Q->stream;
    if (!Q || !slot_out) return fail(HG_ERR_INVALID, "hg_pool_add: pool and slot are required");
    const size_t n = prep.n;
    for (auto &r : prep.rows)
        if (r.size() > Q->cap_s || (Q->bcnt && r.size() > kMaxBondsPerParticle))
            return fail(HG_ERR_CAPACITY, "hg_pool_add: a particle has " + std::to_string(r.size()) +
                                             " bonds, pair capacity is " + std::to_string(Q->cap_s));
    int32_t slot = -1;
    for (size_t s = 0; s < Q->S; s++)
        if (!Q->active[s]) {
            slot = int32_t(s);
            break;
        }
    if (slot < 0) return fail(HG_ERR_CAPACITY, "hg_pool_add: every system slot is in use");
    auto it = Q->free_ranges.begin();
    for (; it != Q->free_ranges.end(); ++it)
        if (it->second >= n) break;
    if (it == Q->free_ranges.end()) return fail(HG_ERR_CAPACITY, "hg_pool_add: no free particle range of that size");
    const uint32_t offset = it->first;
    const uint32_t len = it->second;
    Q->free_ranges.erase(it);
    if (len > n) Q->free_ranges[offset + uint32_t(n)] = len - uint32_t(n);
    Q->high_water = std::max<uint32_t>(Q->high_water, offset + uint32_t(n));

    double *dst[4] = {Q->x, Q->v, Q->th, Q->w};
    for (int f = 0; f < 4; f++)
        HG_HIP(hipMemcpyAsync(dst[f] + 4 * size_t(offset), prep.q4[f].data(), prep.q4[f].size() * 8,
                              hipMemcpyHostToDevice, cs));
    HG_HIP(launch_zero_f64(Q->a + 4 * size_t(offset), 4 * n, cs));
    HG_HIP(launch_zero_f64(Q->al + 4 * size_t(offset), 4 * n, cs));
    std::vector<uint32_t> own(n, uint32_t(slot));
    HG_HIP(hipMemcpyAsync(Q->owner + offset, own.data(), n * 4, hipMemcpyHostToDevice, cs));
    std::vector<uint32_t> pj, cnt;
    if (Q->cap_s) {
        pj.assign(size_t(Q->cap_s) * n, kNoEntry);
        cnt.assign(n, 0u);
        for (size_t i = 0; i < prep.rows.size(); i++) {
            cnt[i] = uint32_t(prep.rows[i].size());
            for (size_t s = 0; s < prep.rows[i].size(); s++)
                pj[s * n + i] = (prep.rows[i][s] & kBondBit) | (offset + (prep.rows[i][s] & kIdxMask));
        }
        HG_HIP(hipMemcpy2DAsync(Q->pj[0] + offset, Q->P * 4, pj.data(), n * 4, n * 4, Q->cap_s,
                                hipMemcpyHostToDevice, cs));
        HG_HIP(hipMemcpyAsync(Q->pcnt[0] + offset, cnt.data(), n * 4, hipMemcpyHostToDevice, cs));
        k_zero_rows_f64<<<256, 256, 0, cs>>>(Q->ps[0], size_t(Q->P) * kSpringRec, size_t(offset) * kSpringRec,
                                                     n * kSpringRec, Q->cap_s);
        HG_HIP(hipGetLastError());
    }
    if (Q->cap_n) HG_HIP(launch_zero_u32(Q->ncnt + offset, n, cs));
    // the host buffers above are read by the copies: wait before they go
    HG_HIP(hipStreamSynchronize(cs));
    Q->meta[slot] = pool_meta{offset, uint32_t(n), 0, 0, 0, 1, uint32_t(slot), 0};
    Q->step_index[slot] = 0;
    Q->t[slot] = 0.0;
    Q->active[slot] = 1;
    Q->fault[slot] = 0;
    Q->bonds[slot] = std::move(prep.bonds);
    Q->skipped[slot] = prep.skipped;
    Q->order_dirty = true;
    Q->meta_dirty = true;
    *slot_out = slot;
    if (Q->bcnt) {  // neck strengths start infinite
        std::vector<double> inf(Q->bonds[slot].size(), std::numeric_limits<double>::infinity());
        PG_TRY(pool_set_necks(Q, slot, inf.data(), cs));
    }
    return HG_OK;
}

}  // namespace hg

namespace {
// hg_pool_add; `given_bonds` (with `given_skipped`) replaces the bond search
// on x0 (a system reloaded from a snapshot keeps the bonds it was built with).
hg_status pool_add_impl(hg_pool *Q, size_t n, const double *x0, const double *v0, const double *theta0,
                        const double *omega0, const std::vector<std::pair<uint32_t, uint32_t>> *given_bonds,
                        size_t given_skipped, int32_t *slot_out) {
    if (!Q || !x0 || !slot_out) return fail(HG_ERR_INVALID, "hg_pool_add: pool, x0 and slot are required");
    pool_prep prep;
    PG_TRY(pool_prepare(Q->p, n, x0, v0, theta0, omega0, given_bonds, given_skipped, prep));
    return pool_commit(Q, prep, slot_out, Q->stream);
}
}  // namespace

extern "C" {

hg_status hg_pool_add(hg_pool *Q, size_t n, const double *x0, const double *v0, const double *theta0,
                      const double *omega0, int32_t *slot_out) {
    return pool_add_impl(Q, n, x0, v0, theta0, omega0, nullptr, 0, slot_out);
}

hg_status hg_pool_set_neck_strengths(hg_pool *Q, int32_t slot, const double *strengths) {
    return pool_set_necks(Q, slot, strengths, Q ? Q->stream : nullptr);
}

}  // extern "C"

namespace hg {

// hg_pool_set_neck_strengths with the copies on stream cs (the copy stream
// while an interval runs: the slot is not in the launch order).
hg_status pool_set_necks(hg_pool *Q, int32_t slot, const double *strengths, hipStream_t cs) {
    PG_TRY(valid_slot(Q, slot));
    if (!strengths) return fail(HG_ERR_INVALID, "strengths is null");
    if (!Q->bcnt) return fail(HG_ERR_INVALID, "hg_pool_set_neck_strengths: the pool's bonds do not break "
                                              "(params.sinter_breaking)");
    const uint32_t off = Q->meta[slot].offset, n = Q->meta[slot].n;
    std::vector<uint32_t> bj(size_t(kMaxBondsPerParticle) * n, kNoEntry), cnt(n, 0);
    std::vector<double> bs(size_t(kMaxBondsPerParticle) * n, 0.0);
    for (size_t b = 0; b < Q->bonds[slot].size(); b++) {
        for (int end = 0; end < 2; end++) {
            const uint32_t i = end ? Q->bonds[slot][b].second : Q->bonds[slot][b].first;
            const uint32_t j = end ? Q->bonds[slot][b].first : Q->bonds[slot][b].second;
            bj[size_t(cnt[i]) * n + i] = off + j;  // arena index, as the pair-state tags
            bs[size_t(cnt[i]) * n + i] = strengths[b];
            cnt[i]++;
        }
    }
    HG_HIP(hipMemcpy2DAsync(Q->bj + off, Q->P * 4, bj.data(), n * 4, n * 4, kMaxBondsPerParticle,
                            hipMemcpyHostToDevice, cs));
    HG_HIP(hipMemcpy2DAsync(Q->bstr + off, Q->P * 8, bs.data(), n * 8, n * 8, kMaxBondsPerParticle,
                            hipMemcpyHostToDevice, cs));
    HG_HIP(hipMemcpyAsync(Q->bcnt + off, cnt.data(), n * 4, hipMemcpyHostToDevice, cs));
    HG_HIP(hipStreamSynchronize(cs));
    return HG_OK;
}

}  // namespace hg

namespace hg {

hg_status pool_release(hg_pool *Q, int32_t slot, hipStream_t cs) {
    PG_TRY(valid_slot(Q, slot));
    const uint32_t off = Q->meta[slot].offset, n = Q->meta[slot].n;
    {
        std::vector<uint32_t> none(n, kNoEntry);
        HG_HIP(hipMemcpyAsync(Q->owner + off, none.data(), n * 4, hipMemcpyHostToDevice, cs));
        HG_HIP(hipStreamSynchronize(cs));
    }
    Q->active[slot] = 0;
    Q->parked[slot] = 0;
    Q->fault[slot] = 0;
    Q->meta[slot] = pool_meta{0, 0, 0, 0, 0, 0, 0, 0};
    Q->bonds[slot].clear();
    Q->order_dirty = true;
    // free the range and coalesce with neighbours
    auto it = Q->free_ranges.emplace(off, n).first;
    auto nx = std::next(it);
    if (nx != Q->free_ranges.end() && it->first + it->second == nx->first) {
        it->second += nx->second;
        Q->free_ranges.erase(nx);
    }
    if (it != Q->free_ranges.begin()) {
        auto pv = std::prev(it);
        if (pv->first + pv->second == it->first) {
            pv->second += it->second;
            Q->free_ranges.erase(it);
        }
    }
    // lower the high-water mark when the top range is free
    auto last = std::prev(Q->free_ranges.end());
    if (last->first + last->second == Q->P) Q->high_water = std::min<uint32_t>(Q->high_water, last->first);
    Q->meta_dirty = true;
    return HG_OK;
}

hg_status pool_read_state(hg_pool *Q, int32_t slot, double *x, double *v, double *theta, double *omega,
                          hipStream_t cs) {
    PG_TRY(valid_slot(Q, slot));
    const size_t off = 4 * size_t(Q->meta[slot].offset);
    const double *src[4] = {Q->x + off, Q->v + off, Q->th + off, Q->w + off};
    double *dst[4] = {x, v, theta, omega};
    return read_fields(Q->stage, src, dst, 4, Q->meta[slot].n, cs);
}

hipStream_t pool_copy_stream(hg_pool *Q) { return Q->stream_c; }

}  // namespace hg

extern "C" {

hg_status hg_pool_remove(hg_pool *Q, int32_t slot) {
    PG_TRY(valid_slot(Q, slot));
    HG_HIP(hipStreamSynchronize(Q->stream));
    return pool_release(Q, slot, Q->stream);
}

}  // extern "C"

namespace hg {

hg_status pool_set_facets(hg_pool *Q, int32_t slot, size_t nf, const double *verts, const double *v_facet,
                          hipStream_t cs) {
    PG_TRY(valid_slot(Q, slot));
    if (nf > Q->MF) return fail(HG_ERR_INVALID, "hg_pool_set_facets: more facets than the pool's max_facets");
    if (nf > 0 && (!verts || !v_facet)) return fail(HG_ERR_INVALID, "hg_pool_set_facets: verts and v_facet required");
    std::vector<facet_dev> F(std::max<size_t>(nf, 1));
    for (size_t f = 0; f < nf; f++) {
        const double *q = verts + 9 * f;
        for (int k = 0; k < 3; k++) F[f].vert[k] = d3{q[3 * k], q[3 * k + 1], q[3 * k + 2]};
        F[f].v_facet = d3{v_facet[3 * f], v_facet[3 * f + 1], v_facet[3 * f + 2]};
        d3 u = F[f].vert[1] - F[f].vert[0], w = F[f].vert[2] - F[f].vert[0];
        F[f].area = 1.0 / 2.0 * norm(cross(u, w));
        F[f].normal = normalized(cross(u, w));
        F[f].pad[0] = F[f].pad[1] = 0.0;
    }
    if (nf > 0) {
        HG_HIP(hipMemcpyAsync(Q->facets + size_t(slot) * Q->MF, F.data(), nf * sizeof(facet_dev),
                              hipMemcpyHostToDevice, cs));
        k_zero_rows_f64<<<256, 256, 0, cs>>>(Q->ss, Q->P, Q->meta[slot].offset, Q->meta[slot].n,
                                                    uint32_t(nf * 9));
        HG_HIP(hipGetLastError());
    }
    HG_HIP(hipStreamSynchronize(cs));
    Q->meta[slot].nf = uint32_t(nf);
    Q->meta[slot].acc_valid = 0;
    Q->meta_dirty = true;
    return HG_OK;
}

}  // namespace hg

extern "C" {

hg_status hg_pool_set_facets(hg_pool *Q, int32_t slot, size_t nf, const double *verts, const double *v_facet) {
    return pool_set_facets(Q, slot, nf, verts, v_facet, Q ? Q->stream : nullptr);
}

namespace {

// How many of the active systems, largest first, take the wide launches: all
// of at least wide_min particles, and as many of the others as the estimates
// below favour (none when wide_min = 0 or the estimate is off).
//
// A step of the wide launches costs a launch's latency or the chip's rate over
// their particles, whichever is more; the chunk kernel's costs its longest
// item (a workgroup goes through its system a particle per thread at a time)
// or the sum of its items over the workgroups. Measured on MI355X, lists of
// 3.9: per-step launches 8 us up to 30,000 particles, then 0.24 ns (mixed) or
// 0.33 ns (FP64) a particle; a round of a 512-thread workgroup 20 us (mixed) or
// 42 us (FP64), of a 256-thread one 12 and 25. So a system of 4,000 particles
// held a launch of 50 steps for 176 us a step (mixed) where the tiles take 8,
// and the chunk kernel's better rate (0.15 ns mixed, the same 0.33 ns in FP64)
// only shows once every workgroup has work: 635,000 particles in 1,024
// systems, mixed, took 206 us a step with the line at 4,096, 128 at 1,536 and
// 166 at 512; 210,000 in 333, FP64, 291 us at 2,048 and 75 all wide.
// With all pairs a round costs 0.5 us a partner and the tiles 0.1 ns a pair at
// 522 particles (0.03 from 3,000 on, and the walk takes over above).
size_t split_order(const hg_pool *Q) {
    const size_t count = Q->order.size();
    if (!Q->wide_min) return 0;
    const bool mixed = Q->p.precision == HG_PRECISION_MIXED, all = Q->p.pair_mode == HG_PAIRS_ALL;
    const double tpb = Q->chunk_tpb, wgs = Q->grid, round_us = mixed ? 0.032 * tpb + 4.0 : 0.068 * tpb + 7.0;
    auto tile_us = [&](double n) { return all ? 1e-4 * n * n : (mixed ? 0.24e-3 : 0.33e-3) * n; };
    auto item_us = [&](double n) { return std::max(1.0, n / tpb) * (all ? 0.5 * n : round_us); };
    // a system smaller than a workgroup shares it with others (lists only)
    auto share_us = [&](double n) { return all || n >= tpb ? item_us(n) : round_us * n / tpb; };
    double chunk = 0.0;
    for (uint32_t s : Q->order) chunk += share_us(Q->meta[s].n);
    size_t best = 0;
    double best_us = 0.0, wide = 0.0;
    for (size_t k = 0; k <= count; k++) {
        const double longest = k < count ? item_us(Q->meta[Q->order[k]].n) : 0.0;
        const bool required = k < count && Q->meta[Q->order[k]].n >= Q->wide_min;
        const bool boundary = k == 0 || k == count || Q->meta[Q->order[k]].n != Q->meta[Q->order[k - 1]].n;
        if (!required && !Q->estimate) return k;
        if (!required && boundary) {
            const double us = (k ? std::max(8.0, wide) : 0.0) + std::max(longest, chunk / wgs);
            if (best_us == 0.0 || us < best_us) {
                best_us = us;
                best = k;
            }
        }
        if (k < count) {
            wide += tile_us(Q->meta[Q->order[k]].n);
            chunk = std::max(0.0, chunk - share_us(Q->meta[Q->order[k]].n));
        }
    }
    return best;
}

// Sorts the active systems largest first, splits off those that take the
// wide launches and uploads the chunk kernel's queue and the wide block map.
hg_status refresh_order(hg_pool *Q) {
    Q->order.clear();
    for (size_t s = 0; s < Q->S; s++)
        if (Q->active[s] && !Q->fault[s] && !Q->parked[s]) Q->order.push_back(uint32_t(s));
    std::stable_sort(Q->order.begin(), Q->order.end(),
                     [&](uint32_t a, uint32_t b) { return Q->meta[a].n > Q->meta[b].n; });
    std::vector<wide_block> map;
    const size_t first_narrow = split_order(Q);
    Q->wide_walk = false;
    if (Q->p.pair_mode == HG_PAIRS_ALL && first_narrow) {
        // tiles take a time per pair, the walk one per particle of the largest
        double pairs = 0.0;
        for (size_t k = 0; k < first_narrow; k++) pairs += double(Q->meta[Q->order[k]].n) * Q->meta[Q->order[k]].n;
        Q->wide_walk = pairs > double(all_pairs_tile_most(Q->p)) * Q->meta[Q->order[0]].n;
    }
    const uint32_t width = Q->wide_walk ? kWalkBlock : uint32_t(tile_width(Q->p.pair_mode));
    for (size_t k = 0; k < first_narrow; k++) {
        const uint32_t s = Q->order[k];
        const pool_meta &M = Q->meta[s];
        for (uint32_t st = 0; st < M.n; st += width)
            map.push_back(wide_block{s, st, M.offset, M.n | (M.cur ? kBondBit : 0u)});
    }
    if (map.size() > Q->wide_map_cap) return fail(HG_ERR_INVALID, "hg_pool_step: wide map overflow");
    Q->narrow_count = uint32_t(Q->order.size() - first_narrow);
    Q->wide_from = first_narrow ? Q->meta[Q->order[first_narrow - 1]].n : 0u;
    Q->wide_blocks = unsigned(map.size());
    // The queue, largest first: each system of at least a workgroup's
    // threads alone, then (neighbour-list mode) the smaller ones packed best
    // fit decreasing: each, in descending size, joins the fullest pack it
    // fits (one particle per thread, at most kMaxPack members), or opens one.
    const bool pack = Q->packing && Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST;
    const uint32_t tpb = uint32_t(Q->chunk_tpb);
    std::vector<uint32_t> slots, packs;
    slots.reserve(Q->narrow_count);
    size_t k = first_narrow;
    for (; k < Q->order.size() && (!pack || Q->meta[Q->order[k]].n >= tpb); k++) {
        packs.push_back(uint32_t(slots.size()) | (1u << 24));
        slots.push_back(Q->order[k]);
    }
    if (k < Q->order.size()) {
        std::vector<std::vector<uint32_t>> bins;
        std::vector<uint32_t> fill;
        std::vector<std::vector<uint32_t>> open(tpb + 1);  // bins with room for a member, by fill
        for (; k < Q->order.size(); k++) {
            const uint32_t s = Q->order[k], n = Q->meta[s].n;
            uint32_t b = ~0u;
            for (uint32_t f = tpb - n; f >= 1 && b == ~0u; f--)
                if (!open[f].empty()) {
                    b = open[f].back();
                    open[f].pop_back();
                }
            if (b == ~0u) {
                b = uint32_t(bins.size());
                bins.emplace_back();
                fill.push_back(0);
            }
            bins[b].push_back(s);
            fill[b] += n;
            if (bins[b].size() < kMaxPack) open[fill[b]].push_back(b);
        }
        std::vector<uint32_t> idx(bins.size());
        for (uint32_t b = 0; b < idx.size(); b++) idx[b] = b;
        std::stable_sort(idx.begin(), idx.end(), [&](uint32_t a, uint32_t b) { return fill[a] > fill[b]; });
        for (uint32_t b : idx) {
            packs.push_back(uint32_t(slots.size()) | (uint32_t(bins[b].size()) << 24));
            slots.insert(slots.end(), bins[b].begin(), bins[b].end());
        }
    }
    Q->pack_count = uint32_t(packs.size());
    if (Q->narrow_count) {
        HG_HIP(hipMemcpyAsync(Q->order_d, slots.data(), slots.size() * 4, hipMemcpyHostToDevice, Q->stream));
        HG_HIP(hipMemcpyAsync(Q->packs_d, packs.data(), packs.size() * 4, hipMemcpyHostToDevice, Q->stream));
    }
    if (!map.empty())
        HG_HIP(hipMemcpyAsync(Q->wide_map_d, map.data(), map.size() * sizeof(wide_block), hipMemcpyHostToDevice,
                              Q->stream));
    HG_HIP(hipStreamSynchronize(Q->stream));
    Q->order_dirty = false;
    return HG_OK;
}

// Online tuner, in two stages: the chunk kernel's shape (256 threads, two
// workgroups per CU; 512 threads, one: the same waves per SIMD with twice the
// LDS per system), then the launch split: the one in use with the wide launches
// ahead of the chunk kernel or beside it, with room for CUs/8 or CUs/4, and
// thresholds that the estimate may have missed, none and those that divide the
// pool's sizes, without it. Every candidate runs two intervals (the first may
// record a graph); the second one's host-measured time per step is its score.
// Neither choice changes any result, so tuning happens on live steps. While all
// of a pool's systems go wide there is nothing to tune; it goes on once one does
// not.
void tune_splits(hg_pool *Q) {
    Q->tune_cands.clear();
    for (int cus : {0, Q->n_cus / 8, Q->n_cus / 4})
        Q->tune_cands.push_back({Q->asked_min, Q->asked_estimate, cus, Q->chunk_tpb, Q->wg_per_cu});
    const uint32_t largest = Q->order.empty() ? 0u : Q->meta[Q->order.front()].n;
    for (uint32_t wm : {0u, 1024u, 2048u, 4096u, 8192u})
        if (wm <= largest && (wm != Q->asked_min || Q->asked_estimate))
            Q->tune_cands.push_back({wm, false, 0, Q->chunk_tpb, Q->wg_per_cu});
    Q->tune_stage = 1;
    Q->tune_scores.assign(Q->tune_cands.size(), 0.0);
    Q->tune_pos = 0;
    Q->tune_phase = TUNE_RUNNING;
}

hg_status tune_begin(hg_pool *Q) {
    if (Q->wide_min != Q->asked_min || Q->estimate != Q->asked_estimate) {  // an earlier tuning's choice
        Q->wide_min = Q->asked_min;
        Q->estimate = Q->asked_estimate;
        PG_TRY(refresh_order(Q));
    }
    if (Q->narrow_count == 0) {
        Q->tune_phase = TUNE_IDLE;
        return HG_OK;
    }
    Q->tune_cands = {{Q->wide_min, Q->estimate, Q->wide_cus, 256, 2}, {Q->wide_min, Q->estimate, Q->wide_cus, 512, 1}};
    Q->tune_stage = 0;
    Q->tune_scores.assign(Q->tune_cands.size(), 0.0);
    Q->tune_pos = 0;
    Q->tune_phase = TUNE_RUNNING;
    return HG_OK;
}

void tune_apply(hg_pool *Q, const hg_pool::tune_cand &c) {
    if (Q->wide_min != c.wide_min || Q->estimate != c.estimate) Q->order_dirty = true;
    Q->wide_min = c.wide_min;
    Q->estimate = c.estimate;
    Q->wide_cus = c.wide_cus;
    if (Q->chunk_tpb != c.tpb) Q->order_dirty = true;  // the packs follow the threads per workgroup
    Q->chunk_tpb = c.tpb;
    set_chunk_wgs(Q, c.wgs);
}

void tune_select(hg_pool *Q) { tune_apply(Q, Q->tune_cands[Q->tune_pos / 2]); }

void tune_record(hg_pool *Q, double seconds_per_step) {
    if (Q->tune_pos % 2 == 1) Q->tune_scores[Q->tune_pos / 2] = seconds_per_step;
    if (++Q->tune_pos < 2 * Q->tune_cands.size()) return;
    size_t best = 0;
    for (size_t k = 1; k < Q->tune_cands.size(); k++)
        if (Q->tune_scores[k] < Q->tune_scores[best]) best = k;
    tune_apply(Q, Q->tune_cands[best]);
    Q->order_dirty = true;
    if (Q->tune_stage == 0)
        tune_splits(Q);
    else
        Q->tune_phase = TUNE_DONE;
}
}  // namespace

}  // extern "C"

namespace hg {

hg_status pool_begin(hg_pool *Q, double dt, uint64_t max_len, uint32_t rebuild_every, uint32_t *len_out) {
    *len_out = 0;
    if (Q->fl.active) return fail(HG_ERR_INVALID, "pool: an interval is already queued");
    if (Q->order_dirty) PG_TRY(refresh_order(Q));
    if (Q->order.empty() || max_len == 0) return HG_OK;
    if (Q->tune_phase == TUNE_START || Q->tune_phase == TUNE_IDLE) PG_TRY(tune_begin(Q));
    if (Q->tune_phase == TUNE_RUNNING) {
        tune_select(Q);
        if (Q->order_dirty) PG_TRY(refresh_order(Q));
    }
    const bool nl = Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST;
    const bool cadence = nl && rebuild_every;
    const pool_view V = make_pool_view(Q);
    const double half = dt / 2.0;
    // one launch runs every system up to the nearest step at which any of
    // them is due for a rebuild, as hg_step does per system
    uint64_t len64 = std::min<uint64_t>(cadence ? rebuild_every : 2000, max_len);
    if (cadence)
        for (uint32_t s : Q->order) len64 = std::min<uint64_t>(len64, rebuild_every - Q->step_index[s] % rebuild_every);
    const uint32_t len = uint32_t(len64);
    const uint32_t count = Q->narrow_count;
    const unsigned grid = unsigned(std::min<uint64_t>(Q->pack_count, uint64_t(Q->grid)));
    bool any_wide_initial = false;
    for (size_t k = 0; k < Q->order.size() - count; k++) any_wide_initial |= !Q->meta[Q->order[k]].acc_valid;
    const auto t_interval = std::chrono::steady_clock::now();
    // The interval's device work is queued without waiting in between: the
    // meta (with the rebuild flags of the systems due) goes up from pinned
    // memory, the rebuild follows on the pool's stream, and the wide launches
    // on the second stream wait for it by an event.
    HG_HIP(hipEventRecord(Q->evb[0], Q->stream));
    bool rebuilt = false;
    if (nl)
        for (uint32_t s : Q->order) {
            const bool due = Q->meta[s].rebuild || (cadence && Q->step_index[s] % rebuild_every == 0);
            Q->meta[s].rebuild = due ? 1u : 0u;
            rebuilt |= due;
        }
    std::memcpy(Q->meta_pinned, Q->meta.data(), Q->S * sizeof(pool_meta));
    HG_HIP(hipMemcpyAsync(Q->meta_d, Q->meta_pinned, Q->S * sizeof(pool_meta), hipMemcpyHostToDevice, Q->stream));
    Q->meta_dirty = false;
    if (rebuilt) {
        HG_HIP(hipEventRecord(Q->ev[0], Q->stream));
        PG_TRY(rebuild_due(Q));
        for (uint32_t s : Q->order) Q->meta[s].rebuild = 0;
    }
    HG_HIP(hipEventRecord(Q->ev[1], Q->stream));
    // wide systems: per-step launches on their own CUs, beside the chunk
    // kernel on the others (all CUs go to whichever kind is alone)
    // wide_cus = 0: no split; the wide steps are queued on the pool's stream
    // ahead of the chunk kernel and each kind has the whole GPU in turn
    const bool split = Q->wide_blocks && count && Q->wide_cus > 0;
    hipStream_t sc = Q->stream;
    if (Q->wide_blocks) {
        hipStream_t s2 = split ? Q->stream_w : Q->stream;
        if (split) HG_HIP(hipStreamWaitEvent(Q->stream_w, Q->ev[1], 0));
        HG_HIP(hipEventRecord(Q->wev[0], s2));
        bool wide_facets = false;
        for (size_t k = 0; k < Q->order.size() - count; k++) wide_facets |= Q->meta[Q->order[k]].nf > 0;
        if (any_wide_initial) {
            HG_HIP(Q->wide_walk
                       ? launch_walk(Q->p, V, Q->wide_map_d, Q->wide_blocks, -1, s2)
                       : launch_tile(Q->p, V, V, Q->wide_map_d, Q->wide_blocks, TILE_FORCE, wide_facets, half, dt, s2));
            Q->last_wide_launches++;
        }
        pool_view VB = V;
        VB.x = Q->xb;
        VB.v = Q->vb;
        VB.w = Q->wb;
        VB.facets = Q->facets_b;
        // the interval's launches: recorded once into a HIP graph per
        // (interval length, dt, wide set, facets or not) and replayed;
        // launched one by one when graphs are off or no system is wide by the
        // threshold: the host queues a launch in 2.7 us and a step takes 8, and
        // a program that copies through the default stream in another thread
        // while a pool of small systems steps must not meet a recording
        auto enqueue = [&](hipStream_t st_) {
            return Q->wide_walk ? launch_walk_steps(Q->p, V, Q->wide_map_d, Q->wide_blocks, len, half, dt, st_)
                                : launch_tile_steps(Q->p, V, VB, Q->wide_map_d, Q->wide_blocks, len, wide_facets, half,
                                                    dt, st_);
        };
        if (Q->wide_graph && Q->meta[Q->order[0]].n >= Q->wide_min) {
            if (!Q->wg_exec || Q->wg_len != len || Q->wg_dt != dt || Q->wg_blocks != Q->wide_blocks ||
                Q->wg_facets != wide_facets || Q->wg_walk != Q->wide_walk) {
                if (Q->wg_exec) HG_HIP(hipGraphExecDestroy(Q->wg_exec));
                Q->wg_exec = nullptr;
                hipGraph_t graph = nullptr;
                HG_HIP(hipStreamBeginCapture(Q->stream_w, hipStreamCaptureModeThreadLocal));
                const hipError_t ec = enqueue(Q->stream_w);
                const hipError_t ee = hipStreamEndCapture(Q->stream_w, &graph);
                HG_HIP(ec);
                HG_HIP(ee);
                const hipError_t ei = hipGraphInstantiate(&Q->wg_exec, graph, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph);
                HG_HIP(ei);
                Q->wg_len = len;
                Q->wg_facets = wide_facets;
                Q->wg_walk = Q->wide_walk;
                Q->wg_dt = dt;
                Q->wg_blocks = Q->wide_blocks;
            }
            HG_HIP(hipGraphLaunch(Q->wg_exec, s2));
        } else {
            HG_HIP(enqueue(s2));
        }
        Q->last_wide_launches += Q->wide_walk ? 2 * len + 1 : len + 1;
        HG_HIP(hipEventRecord(Q->wev[1], s2));
    }
    if (count) {
        const unsigned g = split ? std::min(grid, unsigned(Q->wg_per_cu * (Q->n_cus - Q->wide_cus))) : grid;
        HG_HIP(launch_zero_u32(Q->counter_d, 1, sc));
        HG_HIP(hipEventRecord(Q->ev[2], sc));
        bool facets = false;
        for (size_t k = Q->order.size() - count; k < Q->order.size(); k++) facets |= Q->meta[Q->order[k]].nf > 0;
        const chunk_launch c{Q->order_d, Q->packs_d, Q->pack_count, Q->counter_d, len,
                             dt,         g,          Q->lds_cap,    facets,       Q->chunk_tpb};
        hipError_t e = nl ? launch_chunk_p<HG_PAIRS_NEIGHBOR_LIST>(Q->p, V, c, sc)
                          : launch_chunk_p<HG_PAIRS_ALL>(Q->p, V, c, sc);
        HG_HIP(e);
        HG_HIP(hipEventRecord(Q->ev[3], sc));
    }
    if (split) HG_HIP(hipStreamWaitEvent(Q->stream, Q->wev[1], 0));
    HG_HIP(hipEventRecord(Q->evb[1], Q->stream));
    HG_HIP(launch_copy_words(Q->flags, Q->flags_host, FLAG_COUNT, Q->stream));
    Q->fl.active = true;
    Q->fl.len = len;
    Q->fl.count = count;
    Q->fl.rebuilt = rebuilt;
    Q->fl.wide = Q->wide_blocks != 0;
    Q->fl.dt = dt;
    Q->fl.t0 = t_interval;
    *len_out = len;
    return HG_OK;
}

hg_status pool_end(hg_pool *Q, std::vector<int32_t> &faulted) {
    if (!Q->fl.active) return HG_OK;
    Q->fl.active = false;
    const uint32_t len = Q->fl.len;
    const double dt = Q->fl.dt;
    HG_HIP(hipStreamSynchronize(Q->stream));
    // host mirror of what the kernels did to each system, before any fault is
    // read, so that the systems that go on keep a true mirror
    // the first ones are wide; tiles update their tables in place
    const size_t in_place = Q->wide_walk ? 0 : Q->order.size() - Q->fl.count;
    for (size_t k = 0; k < Q->order.size(); k++) {
        const uint32_t s = Q->order[k];
        pool_meta &M = Q->meta[s];
        if (Q->cap_s && k >= in_place) {
            if (!M.acc_valid) M.cur ^= 1u;
            M.cur ^= (len & 1u);
        }
        M.acc_valid = 1;
        Q->step_index[s] += len;
        for (uint32_t q = 0; q < len; q++) Q->t[s] = Q->t[s] + dt;
    }
    Q->meta_dirty = true;
    PG_TRY(collect_faults(Q, faulted));
    float ms = 0.f;
    if (Q->fl.rebuilt) {
        HG_HIP(hipEventElapsedTime(&ms, Q->ev[0], Q->ev[1]));
        Q->last_rebuild_ms += ms;
    }
    HG_HIP(hipEventElapsedTime(&ms, Q->evb[0], Q->evb[1]));
    Q->last_busy_ms += ms;
    if (Q->fl.count) {
        HG_HIP(hipEventElapsedTime(&ms, Q->ev[2], Q->ev[3]));
        Q->last_chunk_ms += ms;
        Q->last_chunks++;
        Q->last_chunk_steps += len;
    }
    if (Q->fl.wide) {
        HG_HIP(hipEventElapsedTime(&ms, Q->wev[0], Q->wev[1]));
        Q->last_wide_ms += ms;
    }
    if (Q->tune_phase == TUNE_RUNNING)
        tune_record(Q, std::chrono::duration<double>(std::chrono::steady_clock::now() - Q->fl.t0).count() / len);
    return HG_OK;
}

hg_status pool_fault_status(hg_pool *Q, const std::vector<int32_t> &faulted, const char *where) {
    if (faulted.empty()) return HG_OK;
    bool numeric = false;
    std::string msg = std::string(where) + ": stopped system";
    msg += faulted.size() > 1 ? "s" : "";
    for (int32_t s : faulted) {
        const int f = Q->fault[s];
        numeric |= (f & HG_FAULT_NUMERIC) != 0;
        msg += " " + std::to_string(s) + " (";
        std::string why;
        if (f & HG_FAULT_NEIGHBOR_CAPACITY)
            why += "neighbour list needs " + std::to_string(Q->fault_nl_need) + " slots per particle, capacity is " +
                   std::to_string(Q->cap_n);
        if (f & HG_FAULT_PAIR_CAPACITY)
            why += std::string(why.empty() ? "" : "; ") + "pair-state table needs " +
                   std::to_string(Q->fault_pair_need) + " slots per particle, capacity is " + std::to_string(Q->cap_s);
        if (f & HG_FAULT_NUMERIC) why += std::string(why.empty() ? "" : "; ") + "velocity became NaN or infinite";
        msg += why + ")";
    }
    return fail(numeric ? HG_ERR_NUMERIC : HG_ERR_CAPACITY, msg + "; the other systems completed the steps");
}

void pool_reset_profile(hg_pool *Q) {
    Q->last_chunk_ms = Q->last_rebuild_ms = Q->last_wide_ms = Q->last_busy_ms = 0.0;
    Q->last_chunks = Q->last_wide_launches = Q->last_chunk_steps = 0;
}

void pool_park(hg_pool *Q, int32_t slot) {
    Q->parked[slot] = 1;
    Q->order_dirty = true;
}

}  // namespace hg

extern "C" {

hg_status hg_pool_step(hg_pool *Q, double dt, uint64_t nsteps, uint32_t rebuild_every) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    pool_reset_profile(Q);
    if (nsteps == 0) return HG_OK;
    std::vector<int32_t> faulted;  // systems that stopped during this call
    for (uint64_t done = 0; done < nsteps;) {
        uint32_t len = 0;
        PG_TRY(pool_begin(Q, dt, nsteps - done, rebuild_every, &len));
        if (len == 0) break;
        PG_TRY(pool_end(Q, faulted));
        done += len;
    }
    return pool_fault_status(Q, faulted, "hg_pool_step");  // the next pool_begin uploads the meta
}

hg_status hg_pool_fault(hg_pool *Q, int32_t slot, int *fault) {
    PG_TRY(valid_slot(Q, slot));
    if (!fault) return fail(HG_ERR_INVALID, "hg_pool_fault: fault is required");
    *fault = Q->fault[slot];
    return HG_OK;
}

hg_status hg_pool_set_wide_threshold(hg_pool *Q, size_t wide_min) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (wide_min > 0xffffffffu) wide_min = 0;
    Q->asked_min = uint32_t(wide_min);
    Q->wide_min = Q->asked_min;
    Q->estimate = Q->asked_estimate;  // not an earlier tuning's
    Q->order_dirty = true;
    return HG_OK;
}

hg_status hg_pool_autotune(hg_pool *Q, int enable) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    Q->tune_phase = enable ? TUNE_START : TUNE_OFF;
    return HG_OK;
}

hg_status hg_pool_get_tuning(hg_pool *Q, size_t *wide_min, int *wide_cus, int *tuned) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (wide_min) *wide_min = Q->wide_min;
    if (wide_cus) *wide_cus = Q->wide_cus;
    if (tuned) *tuned = Q->tune_phase == TUNE_DONE || Q->tune_phase == TUNE_IDLE ? 1 : 0;
    return HG_OK;
}

hg_status hg_pool_set_split_estimate(hg_pool *Q, int enable) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    Q->asked_estimate = enable != 0;
    Q->wide_min = Q->asked_min;
    Q->estimate = Q->asked_estimate;
    Q->order_dirty = true;
    return HG_OK;
}

hg_status hg_pool_get_split(hg_pool *Q, size_t *wide_from, int *estimated) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (wide_from) *wide_from = Q->wide_from;
    if (estimated) *estimated = Q->estimate ? 1 : 0;
    return HG_OK;
}

hg_status hg_pool_get_chunk_shape(hg_pool *Q, int *threads, int *wg_per_cu) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (threads) *threads = Q->chunk_tpb;
    if (wg_per_cu) *wg_per_cu = Q->wg_per_cu;
    return HG_OK;
}

hg_status hg_pool_set_wide_graph(hg_pool *Q, int enable) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    Q->wide_graph = enable != 0;
    return HG_OK;
}

hg_status hg_pool_set_packing(hg_pool *Q, int enable) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (Q->packing != (enable != 0)) Q->order_dirty = true;
    Q->packing = enable != 0;
    return HG_OK;
}

hg_status hg_pool_set_chunk_shape(hg_pool *Q, int threads, int wg_per_cu) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (threads != 256 && threads != 512) return fail(HG_ERR_INVALID, "hg_pool_set_chunk_shape: threads 256 or 512");
    if (wg_per_cu < 1 || wg_per_cu > 2048 / threads)
        return fail(HG_ERR_INVALID, "hg_pool_set_chunk_shape: wg_per_cu 1.." + std::to_string(2048 / threads));
    if (Q->chunk_tpb != threads) Q->order_dirty = true;
    Q->chunk_tpb = threads;
    set_chunk_wgs(Q, wg_per_cu);
    return HG_OK;
}

hg_status hg_pool_set_wide_cus(hg_pool *Q, int wide_cus) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (wide_cus < 0 || wide_cus >= Q->n_cus)
        return fail(HG_ERR_INVALID, "hg_pool_set_wide_cus: need 0 <= wide_cus < " + std::to_string(Q->n_cus));
    Q->wide_cus = wide_cus;
    return HG_OK;
}

hg_status hg_pool_last_busy(hg_pool *Q, double *busy_ms) {
    if (!Q || !busy_ms) return fail(HG_ERR_INVALID, "pool and busy_ms are required");
    *busy_ms = Q->last_busy_ms;
    return HG_OK;
}

hg_status hg_pool_last_wide_profile(hg_pool *Q, double *wide_ms, uint64_t *launches) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (wide_ms) *wide_ms = Q->last_wide_ms;
    if (launches) *launches = Q->last_wide_launches;
    return HG_OK;
}

hg_status hg_pool_get_state(hg_pool *Q, int32_t slot, double *x, double *v, double *theta, double *omega) {
    return pool_read_state(Q, slot, x, v, theta, omega, Q ? Q->stream : nullptr);
}

hg_status hg_pool_energy(hg_pool *Q, int32_t slot, double mass, double inertia, double *out) {
    PG_TRY(valid_slot(Q, slot));
    if (!out) return fail(HG_ERR_INVALID, "hg_pool_energy: out is required");
    const pool_meta &M = Q->meta[slot];
    const bool nl = Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST;
    if (nl && M.rebuild)
        return fail(HG_ERR_INVALID, "hg_pool_energy: the system is listed by its first step; step it first");
    if (M.n > Q->energy_cap) {
        if (Q->energy) {
            auto it = std::find(Q->allocations.begin(), Q->allocations.end(), static_cast<void *>(Q->energy));
            if (it != Q->allocations.end()) Q->allocations.erase(it);
            HG_HIP(hipFree(Q->energy));
            Q->energy = nullptr;
            Q->energy_cap = 0;
        }
        PG_TRY(palloc(Q, &Q->energy, size_t(8) * M.n));
        Q->energy_cap = M.n;
    }
    double *terms = Q->energy;
    const energy_view E = pool_energy_view(Q, M);
    std::vector<double> h(size_t(8) * M.n);
    hipError_t e = launch_energy(Q->p, E, mass, inertia, terms, Q->stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(h.data(), terms, h.size() * sizeof(double), hipMemcpyDeviceToHost, Q->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(Q->stream);
    HG_HIP(e);
    sum_energy(h.data(), M.n, out);
    return HG_OK;
}

hg_status hg_pool_energy_noalloc(hg_pool *Q, int32_t slot, double mass, double inertia, double *out) {
    PG_TRY(valid_slot(Q, slot));
    if (!out) return fail(HG_ERR_INVALID, "hg_pool_energy_noalloc: out is required");
    const pool_meta &M = Q->meta[slot];
    if (M.n > kNoAllocParticles)
        return fail(HG_ERR_CAPACITY, "hg_pool_energy_noalloc: " + std::to_string(M.n) + " particles exceed its " +
                                         std::to_string(kNoAllocParticles) + "; use hg_pool_energy");
    if (Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST && M.rebuild)
        return fail(HG_ERR_INVALID, "hg_pool_energy_noalloc: the system is listed by its first step; step it first");
    double *scr = nullptr;
    PG_TRY(noalloc_scratch(Q->device, &scr));
    double *sums = scr + 8 * kNoAllocParticles;
    hipError_t e = launch_energy(Q->p, pool_energy_view(Q, M), mass, inertia, scr, Q->stream);
    if (e == hipSuccess) {
        k_energy_sum<<<1, 64, 0, Q->stream>>>(scr, M.n, sums);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(out, sums, 8 * sizeof(double), hipMemcpyDeviceToHost, Q->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(Q->stream);
    HG_HIP(e);
    return HG_OK;
}

hg_status hg_pool_get_accelerations(hg_pool *Q, int32_t slot, double *a, double *alpha) {
    PG_TRY(valid_slot(Q, slot));
    const size_t off = 4 * size_t(Q->meta[slot].offset);
    const double *src[2] = {Q->a + off, Q->al + off};
    double *dst[2] = {a, alpha};
    return read_fields(Q->stage, src, dst, 2, Q->meta[slot].n, Q->stream);
}

hg_status hg_pool_get_neighbors(hg_pool *Q, int32_t slot, uint64_t *offsets, uint32_t *idx, size_t cap,
                                size_t *total) {
    PG_TRY(valid_slot(Q, slot));
    if (!offsets) return fail(HG_ERR_INVALID, "offsets is required");
    if (!Q->cap_n) return fail(HG_ERR_INVALID, "pool has no neighbour lists");
    const uint32_t off = Q->meta[slot].offset, n = Q->meta[slot].n;
    std::vector<uint32_t> nb(size_t(Q->cap_n) * n), cnt(n);
    PG_TRY(download_rows(Q, Q->nb, off, n, Q->cap_n, nb.data()));
    PG_TRY(download_rows(Q, Q->ncnt, off, n, 1, cnt.data()));
    size_t tot = 0;
    for (uint32_t i = 0; i < n; i++) {
        offsets[i] = tot;
        for (uint32_t k = 0; k < cnt[i]; k++) {
            if (idx && tot < cap) idx[tot] = nb[size_t(k) * n + i] - off;
            tot++;
        }
    }
    offsets[n] = tot;
    if (total) *total = tot;
    return HG_OK;
}

hg_status hg_pool_get_springs(hg_pool *Q, int32_t slot, int which, uint32_t *ij, double *springs, size_t cap,
                              size_t *total) {
    PG_TRY(valid_slot(Q, slot));
    if (total) *total = 0;
    if (!Q->cap_s) return HG_OK;
    const uint32_t off = Q->meta[slot].offset, n = Q->meta[slot].n, cur = Q->meta[slot].cur;
    std::vector<uint32_t> pj(size_t(Q->cap_s) * n), cnt(n);
    std::vector<double> ps(size_t(Q->cap_s) * kSpringRec * n);
    PG_TRY(download_rows(Q, Q->pj[cur], off, n, Q->cap_s, pj.data()));
    PG_TRY(download_rows(Q, Q->ps[cur], off, n, Q->cap_s, ps.data(), kSpringRec));
    PG_TRY(download_rows(Q, Q->pcnt[cur], off, n, 1, cnt.data()));
    size_t tot = 0;
    for (uint32_t i = 0; i < n; i++)
        for (uint32_t s = 0; s < cnt[i]; s++) {
            const uint32_t tag = pj[size_t(s) * n + i];
            if (((tag & kBondBit) != 0) != (which == 1)) continue;
            if (tot < cap) {
                if (ij) {
                    ij[2 * tot] = i;
                    ij[2 * tot + 1] = (tag & kIdxMask) - off;
                }
                if (springs)
                    for (int c = 0; c < 9; c++) springs[9 * tot + c] = ps[(size_t(s) * n + i) * kSpringRec + c];
            }
            tot++;
        }
    if (total) *total = tot;
    return HG_OK;
}

hg_status hg_pool_get_bonds(hg_pool *Q, int32_t slot, uint32_t *pairs, size_t cap, size_t *nbonds,
                            size_t *nskipped) {
    PG_TRY(valid_slot(Q, slot));
    const auto &B = Q->bonds[slot];
    for (size_t b = 0; pairs && b < B.size() && b < cap; b++) {
        pairs[2 * b] = B[b].first;
        pairs[2 * b + 1] = B[b].second;
    }
    if (nbonds) *nbonds = B.size();
    if (nskipped) *nskipped = Q->skipped[slot];
    return HG_OK;
}

hg_status hg_pool_info(hg_pool *Q, int32_t slot, size_t *n, double *t, uint64_t *step_index) {
    PG_TRY(valid_slot(Q, slot));
    if (n) *n = Q->meta[slot].n;
    if (t) *t = Q->t[slot];
    if (step_index) *step_index = Q->step_index[slot];
    return HG_OK;
}

hg_status hg_pool_last_step_profile(hg_pool *Q, double *chunk_ms, double *rebuild_ms, uint64_t *chunks,
                                    uint64_t *chunk_steps) {
    if (!Q) return fail(HG_ERR_INVALID, "pool is null");
    if (chunk_ms) *chunk_ms = Q->last_chunk_ms;
    if (rebuild_ms) *rebuild_ms = Q->last_rebuild_ms;
    if (chunks) *chunks = Q->last_chunks;
    if (chunk_steps) *chunk_steps = Q->last_chunk_steps;
    return HG_OK;
}

}  // extern "C"

namespace {
template <typename T>
hg_status upload_rows(hg_pool *Q, T *dev, uint32_t offset, uint32_t n, uint32_t rows, const std::vector<T> &host,
                      size_t width = 1) {
    if (rows == 0 || n == 0) return HG_OK;
    const size_t row = n * width * sizeof(T);
    HG_HIP(hipMemcpy2DAsync(dev + offset * width, Q->P * width * sizeof(T), host.data(), row, row, rows,
                            hipMemcpyHostToDevice, Q->stream));
    HG_HIP(hipStreamSynchronize(Q->stream));
    return HG_OK;
}
}  // namespace

extern "C" {

hg_status hg_pool_save(hg_pool *Q, int32_t slot, void *buf, size_t cap, size_t *size) {
    PG_TRY(valid_slot(Q, slot));
    if (!size) return fail(HG_ERR_INVALID, "hg_pool_save: size is required");
    const pool_meta &M = Q->meta[slot];
    const uint32_t off = M.offset, n = M.n, cur = M.cur;
    snapshot z;
    z.p = Q->p;
    z.n = n;
    z.t = Q->t[slot];
    z.step_index = Q->step_index[slot];
    z.acc_valid = M.acc_valid;
    const bool nl = Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST;
    z.needs_rebuild = nl && M.rebuild ? 1u : 0u;
    const double *fields[6] = {Q->x, Q->v, Q->th, Q->w, Q->a, Q->al};
    std::vector<double> *dst[6] = {&z.x, &z.v, &z.th, &z.w, &z.a, &z.al};
    for (int f = 0; f < 6; f++) {
        std::vector<double> q4(4 * size_t(n));
        PG_TRY(download_rows(Q, fields[f] + 4 * size_t(off), 0, n, 1, q4.data(), 4));
        *dst[f] = pack3(q4, n);
    }
    if (nl && !M.rebuild) {
        std::vector<uint32_t> nb(size_t(Q->cap_n) * n);
        z.has_nl = true;
        z.nl_count.resize(n);
        PG_TRY(download_rows(Q, Q->nb, off, n, Q->cap_n, nb.data()));
        PG_TRY(download_rows(Q, Q->ncnt, off, n, 1, z.nl_count.data()));
        rows_to_csr(nb.data(), z.nl_count.data(), n, 1, 1, z.nl_ids);
        shift_ids(z.nl_ids, off);
    }
    if (Q->cap_s) {
        std::vector<uint32_t> pj(size_t(Q->cap_s) * n);
        std::vector<double> ps(size_t(Q->cap_s) * kSpringRec * n);
        z.has_table = true;
        z.pt_count.resize(n);
        PG_TRY(download_rows(Q, Q->pj[cur], off, n, Q->cap_s, pj.data()));
        PG_TRY(download_rows(Q, Q->ps[cur], off, n, Q->cap_s, ps.data(), kSpringRec));
        PG_TRY(download_rows(Q, Q->pcnt[cur], off, n, 1, z.pt_count.data()));
        rows_to_csr(pj.data(), z.pt_count.data(), n, 1, 1, z.pt_tags);
        rows_to_csr(ps.data(), z.pt_count.data(), n, kSpringRec, 9, z.pt_springs);
        shift_ids(z.pt_tags, off);
    }
    for (auto &b : Q->bonds[slot]) {
        z.bonds.push_back(b.first);
        z.bonds.push_back(b.second);
    }
    z.skipped = Q->skipped[slot];
    z.nf = M.nf;
    if (M.nf > 0) {
        z.facets.resize(M.nf);
        z.ss.resize(size_t(M.nf) * 9 * n);
        HG_HIP(hipMemcpyAsync(z.facets.data(), Q->facets + size_t(slot) * Q->MF, M.nf * sizeof(facet_dev),
                              hipMemcpyDeviceToHost, Q->stream));
        HG_HIP(hipStreamSynchronize(Q->stream));
        PG_TRY(download_rows(Q, Q->ss, off, n, M.nf * 9, z.ss.data()));
    }
    if (Q->bstr) {
        std::vector<uint32_t> bj(size_t(kMaxBondsPerParticle) * n);
        std::vector<double> bs(size_t(kMaxBondsPerParticle) * n);
        z.has_neck = true;
        z.neck_count.resize(n);
        PG_TRY(download_rows(Q, Q->bj, off, n, kMaxBondsPerParticle, bj.data()));
        PG_TRY(download_rows(Q, Q->bstr, off, n, kMaxBondsPerParticle, bs.data()));
        PG_TRY(download_rows(Q, Q->bcnt, off, n, 1, z.neck_count.data()));
        rows_to_csr(bj.data(), z.neck_count.data(), n, 1, 1, z.neck_j);
        rows_to_csr(bs.data(), z.neck_count.data(), n, 1, 1, z.neck_str);
        shift_ids(z.neck_j, off);
    }
    const std::vector<uint8_t> bytes = encode_snapshot(z);
    *size = bytes.size();
    if (!buf) return HG_OK;
    if (cap < bytes.size())
        return fail(HG_ERR_CAPACITY, "hg_pool_save: the snapshot needs " + std::to_string(bytes.size()) + " bytes");
    std::memcpy(buf, bytes.data(), bytes.size());
    return HG_OK;
}

hg_status hg_pool_load(hg_pool *Q, const void *buf, size_t size, int32_t *slot_out) {
    if (!Q || !slot_out) return fail(HG_ERR_INVALID, "hg_pool_load: pool and slot are required");
    snapshot z;
    PG_TRY(decode_snapshot(buf, size, z));
    if (std::memcmp(&z.p, &Q->p, sizeof(hg_params)) != 0)
        return fail(HG_ERR_INVALID, "hg_pool_load: the snapshot was taken with other parameters than the pool's");
    if (z.has_legacy) return fail(HG_ERR_INVALID, "hg_pool_load: pools do not run the legacy sinter_functor");
    if (z.nf > Q->MF) return fail(HG_ERR_INVALID, "hg_pool_load: more facets than the pool's max_facets");
    if ((z.has_nl && max_count(z.nl_count) > Q->cap_n) || (z.has_table && max_count(z.pt_count) > Q->cap_s))
        return fail(HG_ERR_CAPACITY, "hg_pool_load: a row of the snapshot exceeds the pool's capacity");
    const uint32_t n = uint32_t(z.n);
    std::vector<std::pair<uint32_t, uint32_t>> bonds(z.bonds.size() / 2);
    for (size_t b = 0; b < bonds.size(); b++) bonds[b] = {z.bonds[2 * b], z.bonds[2 * b + 1]};
    int32_t slot = -1;
    PG_TRY(pool_add_impl(Q, n, z.x.data(), z.v.data(), z.th.data(), z.w.data(), &bonds, z.skipped, &slot));
    const uint32_t off = Q->meta[slot].offset;
    auto fill = [&]() -> hg_status {
        for (auto [dev, host] : {std::pair<double *, const std::vector<double> *>{Q->a, &z.a}, {Q->al, &z.al}}) {
            std::vector<double> q4(4 * size_t(n), 0.0);
            for (uint32_t i = 0; i < n; i++)
                for (int c = 0; c < 3; c++) q4[4 * size_t(i) + c] = (*host)[3 * size_t(i) + c];
            HG_HIP(hipMemcpyAsync(dev + 4 * size_t(off), q4.data(), q4.size() * 8, hipMemcpyHostToDevice, Q->stream));
            HG_HIP(hipStreamSynchronize(Q->stream));
        }
        pool_meta &M = Q->meta[slot];
        if (z.has_table && Q->cap_s) {
            std::vector<uint32_t> tags = z.pt_tags, pj;
            std::vector<double> ps;
            shift_ids(tags, -int64_t(off));
            csr_to_rows(z.pt_count, tags, n, Q->cap_s, 1, 1, kNoEntry, pj);
            csr_to_rows(z.pt_count, z.pt_springs, n, Q->cap_s, kSpringRec, 9, 0.0, ps);
            M.cur = 0;
            PG_TRY(upload_rows(Q, Q->pj[0], off, n, Q->cap_s, pj));
            PG_TRY(upload_rows(Q, Q->ps[0], off, n, Q->cap_s, ps, kSpringRec));
            PG_TRY(upload_rows(Q, Q->pcnt[0], off, n, 1, z.pt_count));
        }
        if (Q->p.pair_mode == HG_PAIRS_NEIGHBOR_LIST && z.has_nl) {
            std::vector<uint32_t> ids = z.nl_ids, nb;
            shift_ids(ids, -int64_t(off));
            csr_to_rows(z.nl_count, ids, n, Q->cap_n, 1, 1, 0u, nb);
            PG_TRY(upload_rows(Q, Q->nb, off, n, Q->cap_n, nb));
            PG_TRY(upload_rows(Q, Q->ncnt, off, n, 1, z.nl_count));
            M.rebuild = 0;
        }
        if (z.nf > 0) {
            HG_HIP(hipMemcpyAsync(Q->facets + size_t(slot) * Q->MF, z.facets.data(), z.nf * sizeof(facet_dev),
                                  hipMemcpyHostToDevice, Q->stream));
            HG_HIP(hipStreamSynchronize(Q->stream));
            PG_TRY(upload_rows(Q, Q->ss, off, n, z.nf * 9, z.ss));
            M.nf = z.nf;
        }
        if (z.has_neck && Q->bcnt) {
            if (max_count(z.neck_count) > kMaxBondsPerParticle) return fail(HG_ERR_INVALID, "hg_pool_load: bad neck rows");
            std::vector<uint32_t> ids = z.neck_j, bj;
            std::vector<double> bs;
            shift_ids(ids, -int64_t(off));
            csr_to_rows(z.neck_count, ids, n, kMaxBondsPerParticle, 1, 1, kNoEntry, bj);
            csr_to_rows(z.neck_count, z.neck_str, n, kMaxBondsPerParticle, 1, 1, 0.0, bs);
            PG_TRY(upload_rows(Q, Q->bj, off, n, kMaxBondsPerParticle, bj));
            PG_TRY(upload_rows(Q, Q->bstr, off, n, kMaxBondsPerParticle, bs));
            PG_TRY(upload_rows(Q, Q->bcnt, off, n, 1, z.neck_count));
        }
        M.acc_valid = z.acc_valid;
        Q->t[slot] = z.t;
        Q->step_index[slot] = z.step_index;
        Q->meta_dirty = true;
        Q->order_dirty = true;
        return upload_meta(Q);
    };
    const hg_status st = fill();
    if (st != HG_OK) {
        const std::string msg = hg_last_error();
        (void)hg_pool_remove(Q, slot);
        return fail(st, msg);
    }
    *slot_out = slot;
    return HG_OK;
}

}  // extern "C"

// Device code of the pool's stepping kernels: the chunk kernel (one rebuild
// interval of every queued system, a workgroup per system or pack) and the
// per-step launches of large systems. pool_chunk.hip compiles it once per
// binary functor and pair mode; pool.hip queues the launches.
#pragma once

#include <hip/hip_runtime.h>

#include "force_device.h"
#include "hg_internal.h"

namespace hg {


struct pool_view {
    double *x, *v, *th, *w, *a, *al;
    const uint32_t *nb;
    const uint32_t *ncnt;
    uint32_t *pj0, *pj1, *pcnt0, *pcnt1;
    double *ps0, *ps1;
    uint32_t cap_s, cap_n;
    const uint32_t *bj;  // neck-strength lists (see pair_table), null unless bonds break
    const double *bstr;
    const uint32_t *bcnt;
    facet_dev *facets;
    uint32_t max_facets;
    uint32_t facet_steps;  // 0: facets move only through hg_advance_facet
    double *ss;
    const pool_meta *meta;
    size_t stride;
    int *flags;
    int *sflags;  // per-system fault words (HG_FAULT_* bits), indexed by slot
    uint32_t alone;  // wide_block::n of a single system, whose tiles need no map
};

constexpr uint32_t kDefaultWideMin = 2048;
constexpr double kDefaultWideCuFraction = 0.25;
// TUNE_IDLE: nothing to tune until a system takes the chunk kernel
enum { TUNE_OFF = 0, TUNE_START = 1, TUNE_RUNNING = 2, TUNE_DONE = 3, TUNE_IDLE = 4 };

// Per-step launches (tile_step.h): workgroup b carries the particles
// [start, start + tile_width) of the system at [offset, offset + n) of the
// arena; the top bit of n says which half of the pair-state table is the
// system's current one.
struct wide_block {
    uint32_t slot, start, offset, n;
};
constexpr uint32_t kTileThreads = 256;
constexpr int tile_width(int pairs) { return pairs == HG_PAIRS_NEIGHBOR_LIST ? 64 : 1; }
// List positions a tile takes at a time. Their terms take most of its LDS: with
// twelve, an aggregate's longest lists (r_verlet of 3.2 radii) still fit one
// round, and an FP64 tile takes 52 KB, 70 with facets (sixteen: 70 and 90, one
// workgroup to a CU with facets).
constexpr int tile_depth(int pairs) { return pairs == HG_PAIRS_NEIGHBOR_LIST ? 12 : 1024; }
enum { TILE_FORCE = 0, TILE_STEP = 1, TILE_LAST = 2 };

// The launches of one binary functor and pair mode (pool_chunk.hip), by
// Hamaker model, precision, facets and workgroup size.
struct chunk_launch {
    const uint32_t *order, *packs;  // packs[i] = first | count << 24 over the slots in `order`
    uint32_t count;                 // packs
    uint32_t *counter;              // one word, zero
    uint32_t nsteps;
    double dt;
    unsigned grid;
    uint32_t lds_cap;
    bool facets;  // whether any queued system has facets (else the kernel without the facet fold runs)
    int tpb;      // threads per workgroup (256 or 512)
};
template <int BIN, int PAIRS>
hipError_t launch_chunk_b(const hg_params &p, const pool_view &V, const chunk_launch &c, hipStream_t s);
template <int BIN, int PAIRS>
hipError_t launch_tile_b(const hg_params &p, const pool_view &Vi, const pool_view &Vo, const wide_block *map,
                         unsigned blocks, int mode, bool facets, double half, double dt, hipStream_t s);
hipError_t launch_tile_kick(const pool_view &V, const pool_view &Vo, const wide_block *map, unsigned blocks, int pairs,
                            double half, double dt, hipStream_t s);

// One launch of k_tile_step for the parameters' functors (BINs 0..2).
hipError_t launch_tile(const hg_params &p, const pool_view &Vi, const pool_view &Vo, const wide_block *map,
                       unsigned blocks, int mode, bool facets, double half, double dt, hipStream_t s);
// `len` steps of the systems in `map` from V's buffers back into them, x, v
// and omega (and the facets) alternating with VB's: a kick and drift into the
// set from which the last pass reads VB, then a launch per step.
hipError_t launch_tile_steps(const hg_params &p, const pool_view &V, const pool_view &VB, const wide_block *map,
                             unsigned blocks, uint32_t len, bool facets, double half, double dt, hipStream_t s);

// Per-step launches of large all-pairs systems, a lane a particle
// (all_pairs_tile_most): wide_block b carries [start, start + kWalkBlock), the
// pair-state table alternates between its halves as in the chunk kernel.
// pass < 0: the accelerations of the systems that have none.
constexpr uint32_t kWalkBlock = 128;
template <int BIN>
hipError_t launch_walk_b(const hg_params &p, const pool_view &V, const wide_block *map, unsigned blocks, int pass,
                         hipStream_t s);

template <int PAIRS>
inline hipError_t launch_chunk_p(const hg_params &p, const pool_view &V, const chunk_launch &c, hipStream_t s) {
    if (p.binary_model == HG_BINARY_NONE) return launch_chunk_b<HG_BINARY_NONE, PAIRS>(p, V, c, s);
    if (p.binary_model == HG_BINARY_CONTACT) return launch_chunk_b<HG_BINARY_CONTACT, PAIRS>(p, V, c, s);
    if (p.binary_model == HG_BINARY_SINTER) return launch_chunk_b<HG_BINARY_SINTER, PAIRS>(p, V, c, s);
    return hipErrorInvalidValue;
}
// The FP64 pair path's bond constants held in vector registers for a pass
// (as pinned() does for the mixed path): kept as scalars they are spilled and
// re-read lane by lane inside the pair loop.
__device__ __forceinline__ hg_params pinned64(const hg_params &P) {
    hg_params p = P;
    hg_sinter_params &s = p.sinter;
    double *f[] = {&s.k, &s.gamma_n, &s.k_t, &s.gamma_t, &s.k_r, &s.gamma_r,
                   &s.k_o, &s.gamma_o, &s.r_part, &s.mass, &s.inertia, &s.dt};
#pragma unroll
    for (double *q : f) pin_vgpr(*q);
    return p;
}

}  // namespace hg

namespace hg {

namespace {

// Where a running system's particle state lives during a chunk (chosen per
// system from its size and the workgroup's LDS; local index g - offset):
//   STATE_FULL   all of x, v, omega, theta, a, alpha in LDS (18 doubles per
//                particle), read from global memory at the start of the
//                chunk and written back once at its end;
//   STATE_MIRROR x, v, omega copied into LDS (9 doubles per particle) and
//                refreshed by each owner lane in the kick/drift phase, so
//                partner gathers read LDS; the state itself stays global;
//   STATE_POS    x alone copied into LDS (3 doubles per particle) and
//                refreshed likewise: every partner needs its position, only
//                the bonded and overlapping ones (a few of a 3.2r list) its
//                velocities, which then come from global memory;
//   STATE_GLOBAL everything in global memory.
enum { STATE_GLOBAL = 0, STATE_MIRROR = 1, STATE_FULL = 2, STATE_POS = 3 };
#ifndef HG_CHUNK_EAGER
#define HG_CHUNK_EAGER 1
#endif
#ifndef HG_CHUNK_PREFETCH
#define HG_CHUNK_PREFETCH 1
#endif
#ifndef HG_CHUNK_MIN_BLOCKS
#define HG_CHUNK_MIN_BLOCKS 1
#endif
constexpr bool kChunkEager = HG_CHUNK_EAGER, kChunkPrefetch = HG_CHUNK_PREFETCH;
extern __shared__ double pool_lds[];
constexpr uint32_t kPosStride = 3, kMirrorStride = 9, kFullStride = 18;
template <int MODE>
constexpr uint32_t lds_stride() {
    return MODE == STATE_FULL ? kFullStride : (MODE == STATE_MIRROR ? kMirrorStride : kPosStride);
}

template <int MODE>
__device__ __forceinline__ double *lds_rec(uint32_t offset, uint32_t g) {
    return pool_lds + size_t(g - offset) * lds_stride<MODE>();
}
__device__ __forceinline__ d3 lds3(const double *q) { return d3{q[0], q[1], q[2]}; }
__device__ __forceinline__ void sds3(double *q, d3 a) {
    q[0] = a.x;
    q[1] = a.y;
    q[2] = a.z;
}

template <int MODE>
__device__ __forceinline__ d3 load_x(const pool_view &V, uint32_t offset, uint32_t g) {
    if constexpr (MODE == STATE_GLOBAL) return ld3(V.x, g);
    else return lds3(lds_rec<MODE>(offset, g));
}
template <int MODE>
__device__ __forceinline__ void load_vw(const pool_view &V, uint32_t offset, uint32_t g, d3 &v, d3 &w) {
    if constexpr (MODE == STATE_GLOBAL || MODE == STATE_POS) {
        v = ld3(V.v, g);
        w = ld3(V.w, g);
    } else {
        const double *q = lds_rec<MODE>(offset, g);
        v = lds3(q + 3);
        w = lds3(q + 6);
    }
}

template <int MODE>
__device__ __forceinline__ void load_state(const pool_view &V, uint32_t offset, uint32_t g, d3 &x, d3 &v, d3 &w) {
    if constexpr (MODE == STATE_GLOBAL) {
        x = ld3(V.x, g);
        v = ld3(V.v, g);
        w = ld3(V.w, g);
    } else if constexpr (MODE == STATE_POS) {
        x = lds3(lds_rec<MODE>(offset, g));
        v = ld3(V.v, g);
        w = ld3(V.w, g);
    } else {
        const double *q = lds_rec<MODE>(offset, g);
        x = lds3(q);
        v = lds3(q + 3);
        w = lds3(q + 6);
    }
}

template <int MODE>
__device__ __forceinline__ void store_acc(const pool_view &V, uint32_t offset, uint32_t g, d3 a, d3 al) {
    if constexpr (MODE == STATE_FULL) {
        double *q = lds_rec<MODE>(offset, g);
        sds3(q + 12, a);
        sds3(q + 15, al);
    } else {
        st3(V.a, g, a);
        st3(V.al, g, al);
    }
}

// Fills the LDS records of a system at the start of its chunk.
template <int MODE>
__device__ __forceinline__ void lds_fill(const pool_view &V, const pool_meta &M) {
    for (uint32_t g = M.offset + threadIdx.x; g < M.offset + M.n; g += blockDim.x) {
        double *q = lds_rec<MODE>(M.offset, g);
        sds3(q, ld3(V.x, g));
        if constexpr (MODE == STATE_POS) continue;
        sds3(q + 3, ld3(V.v, g));
        sds3(q + 6, ld3(V.w, g));
        if constexpr (MODE == STATE_FULL) {
            sds3(q + 9, ld3(V.th, g));
            sds3(q + 12, ld3(V.a, g));
            sds3(q + 15, ld3(V.al, g));
        }
    }
}

// LDS copy of a neighbour-list system's partner ids for one rebuild interval:
// kmax slots per particle (kmax = the system's longest list), slot k of local
// particle t at lids[k*n + t] as a halfword offset from the system's first
// particle, then the list counts at lids[kmax*n + t]. A system of at most
// 65,535 particles fits the halfwords.
__host__ __device__ inline size_t lds_ids_bytes(uint32_t n, uint32_t kmax) { return size_t(n) * 2 * (kmax + 1); }

__device__ __forceinline__ void lds_ids_fill(const pool_view &V, const pool_meta &M, uint32_t kmax, uint16_t *lids) {
    for (uint32_t t = threadIdx.x; t < M.n; t += blockDim.x) {
        const uint32_t g = M.offset + t, c = V.ncnt[g];
        lids[kmax * M.n + t] = uint16_t(c);
        for (uint32_t k = 0; k < c; k++) lids[k * M.n + t] = uint16_t(V.nb[size_t(k) * V.stride + g] - M.offset);
    }
}

// Largest value of v over the workgroup (s_red: one word per wavefront).
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t *s_red) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, uint32_t(__shfl_xor(int(v), o)));
    if ((threadIdx.x & 63u) == 0) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t r = 0;
    for (uint32_t w = 0; w < (blockDim.x + 63u) / 64u; w++) r = max(r, s_red[w]);
    __syncthreads();
    return r;
}

// Acceleration pass for particles g = g_first, g_first + g_step, ... < g_end
// of system M (a workgroup strides over the whole system; a pack and the walk of
// large all-pairs systems give each thread one particle). With LIDS the partner ids come from the system's
// LDS copy `lids` (lds_ids_fill).
template <int BIN, int HAM, int PAIRS, int PREC, int LDS, bool LIDS = false, bool FAC = true>
__device__ __forceinline__ void pool_force_phase(const hg_params &P, const mixed_consts &MC, const pool_view &V,
                                                 const pool_meta &M, uint32_t cur, const facet_dev *F,
                                                 uint32_t g_first, uint32_t g_end, uint32_t g_step,
                                                 const uint16_t *lids = nullptr, uint32_t kmax = 0) {
    pair_table T;
    T.pj_old = cur ? V.pj1 : V.pj0;
    T.ps_old = cur ? V.ps1 : V.ps0;
    T.pcnt_old = cur ? V.pcnt1 : V.pcnt0;
    T.pj_new = cur ? V.pj0 : V.pj1;
    T.ps_new = cur ? V.ps0 : V.ps1;
    T.pcnt_new = cur ? V.pcnt0 : V.pcnt1;
    T.cap = V.cap_s;
    T.stride = V.stride;
    T.bj = V.bj;
    T.bstr = V.bstr;
    T.bcnt = V.bcnt;
    const uint32_t end = M.offset + M.n;
    for (uint32_t g = g_first; g < g_end; g += g_step) {
        d3 xi, vi, wi;
        load_state<LDS>(V, M.offset, g, xi, vi, wi);
        walker_t<PREC == HG_PRECISION_MIXED && kChunkEager> W;
        if constexpr (BIN != HG_BINARY_NONE) W.init(T, g);
        id_list ids;
        if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST && !LIDS) ids.init(V.nb, V.ncnt, V.stride, g, V.cap_n);
        // listed partners of g through fold(j, xj, vw), in list order: vw
        // gives a partner's velocities when its pair needs them, from LDS or
        // from a global gather made a pair ahead with its position
        auto partners = [&](auto &&fold) {
            auto run = [&](const auto &ids_) {
                if constexpr (LDS == STATE_GLOBAL) {
                    nl_partners<kChunkPrefetch>(
                        ids_, [&](uint32_t j) { return pstate{ld3(V.x, j), ld3(V.v, j), ld3(V.w, j)}; },
                        [&](uint32_t j, const pstate &sj) {
                            fold(j, sj.x, [&](d3 &v, d3 &w) { v = sj.v, w = sj.w; });
                        });
                } else {
                    nl_partners<kChunkPrefetch>(
                        ids_, [&](uint32_t j) { return load_x<LDS>(V, M.offset, j); },
                        [&](uint32_t j, d3 xj) {
                            fold(j, xj, [&](d3 &v, d3 &w) { load_vw<LDS>(V, M.offset, j, v, w); });
                        });
                }
            };
            if constexpr (LIDS) {
                const uint32_t t = g - M.offset;
                run(lds_id_list{lids, M.n, t, M.offset, lids[kmax * M.n + t]});
            } else {
                run(ids);
            }
        };
        auto vw_of = [&](uint32_t j) { return [&V, &M, j](d3 &v, d3 &w) { load_vw<LDS>(V, M.offset, j, v, w); }; };
        if constexpr (PREC == HG_PRECISION_FP64) {
            acc6 acc{zero3(), zero3()};
            const hg_params pp = pinned64(P);
            if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) {
                partners([&](uint32_t j, d3 xj, auto &&vw) { pair_fold_vw<BIN, HAM>(pp, j, xi, vi, wi, xj, vw, W, acc); });
            } else {
                for (uint32_t j = M.offset; j < end; j++) {
                    if (j == g) continue;
                    pair_fold_vw<BIN, HAM>(P, j, xi, vi, wi, load_x<LDS>(V, M.offset, j), vw_of(j), W, acc);
                }
            }
            close_table<BIN>(W, T.pcnt_new, g, V.flags, V.sflags + M.slot);
            if (FAC && M.nf > 0) acc = acc + facet_fold(P, F, int(M.nf), V.ss, V.stride, g, xi, vi, wi);
            store_acc<LDS>(V, M.offset, g, acc.lin, acc.ang);
        } else {
            accf acc{zerof(), zerof()};
            const mixed_consts m = pinned(MC);
            if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) {
                partners([&](uint32_t j, d3 xj, auto &&vw) { pair_fold_mx<BIN, HAM>(m, j, xi, vi, wi, xj, vw, W, acc); });
            } else {
                for (uint32_t j = M.offset; j < end; j++) {
                    if (j == g) continue;
                    pair_fold_mx<BIN, HAM>(MC, j, xi, vi, wi, load_x<LDS>(V, M.offset, j), vw_of(j), W, acc);
                }
            }
            close_table<BIN>(W, T.pcnt_new, g, V.flags, V.sflags + M.slot);
            if (FAC && M.nf > 0) acc = acc + facet_fold_mx(P, MC, F, int(M.nf), V.ss, V.stride, g, xi, vi, wi);
            const d3 a64 = tod(acc.lin), al64 = tod(acc.ang);
            store_acc<LDS>(V, M.offset, g, a64, al64);
        }
    }
}

// Kick (completing the previous step when `pending`), kick, drift; the same
// operations in the same order as k_kick_drift.
template <int LDS>
__device__ __forceinline__ void pool_kick_drift(const pool_view &V, const pool_meta &M, bool pending, double half,
                                                double dt, uint32_t g_first, uint32_t g_end, uint32_t g_step) {
    for (uint32_t g = g_first; g < g_end; g += g_step) {
        double *q = lds_rec<LDS>(M.offset, g);
        d3 vi, wi, ai, ali, x0, th0;
        if constexpr (LDS == STATE_FULL) {
            vi = lds3(q + 3); wi = lds3(q + 6); ai = lds3(q + 12); ali = lds3(q + 15); x0 = lds3(q); th0 = lds3(q + 9);
        } else {
            vi = ld3(V.v, g); wi = ld3(V.w, g); ai = ld3(V.a, g); ali = ld3(V.al, g); x0 = ld3(V.x, g);
            th0 = ld3(V.th, g);
        }
        if (pending) {
            vi = vi + ai * half;
            wi = wi + ali * half;
        }
        vi = vi + ai * half;
        wi = wi + ali * half;
        const d3 xi = x0 + vi * dt;
        const d3 thi = th0 + wi * dt;
        if constexpr (LDS != STATE_FULL) {
            st3(V.x, g, xi);
            st3(V.th, g, thi);
            st3(V.v, g, vi);
            st3(V.w, g, wi);
        }
        if constexpr (LDS != STATE_GLOBAL) sds3(q, xi);
        if constexpr (LDS == STATE_MIRROR || LDS == STATE_FULL) {
            sds3(q + 3, vi);
            sds3(q + 6, wi);
        }
        if constexpr (LDS == STATE_FULL) sds3(q + 9, thi);
    }
}

// Final kick; a system kept wholly in LDS is written back here. A non-finite
// velocity or angular velocity faults the system (HG_FAULT_NUMERIC).
template <int LDS>
__device__ __forceinline__ void pool_final_kick(const pool_view &V, const pool_meta &M, double half,
                                                uint32_t g_first, uint32_t g_end, uint32_t g_step) {
    bool bad = false;
    for (uint32_t g = g_first; g < g_end; g += g_step) {
        d3 vi, wi;
        if constexpr (LDS == STATE_FULL) {
            const double *q = lds_rec<LDS>(M.offset, g);
            const d3 a = lds3(q + 12), al = lds3(q + 15);
            vi = lds3(q + 3) + a * half;
            wi = lds3(q + 6) + al * half;
            st3(V.x, g, lds3(q));
            st3(V.th, g, lds3(q + 9));
            st3(V.a, g, a);
            st3(V.al, g, al);
        } else {
            vi = ld3(V.v, g) + ld3(V.a, g) * half;
            wi = ld3(V.w, g) + ld3(V.al, g) * half;
        }
        st3(V.v, g, vi);
        st3(V.w, g, wi);
        bad |= nonfinite(vi, wi);
    }
    if (bad) {
        atomicOr(&V.flags[FLAG_NUMERIC], 1);
        atomicOr(&V.sflags[M.slot], HG_FAULT_NUMERIC);
    }
}

// All steps of one rebuild interval for one system, by one workgroup. With
// LIDS the system's partner ids (kmax slots per particle) are copied to LDS
// after its state records.
template <int BIN, int HAM, int PAIRS, int PREC, int LDS, bool LIDS, bool FAC>
__device__ __forceinline__ void run_system(const hg_params &P, const mixed_consts &MC, const pool_view &V,
                                           const pool_meta &M, facet_dev *F, uint32_t nsteps, double dt,
                                           uint32_t kmax) {
    const double half = dt / 2.0;
    uint32_t cur = M.cur;
    const uint32_t g0 = M.offset + threadIdx.x, g_end = M.offset + M.n, gs = blockDim.x;
    if constexpr (LDS != STATE_GLOBAL) lds_fill<LDS>(V, M);
    uint16_t *lids = nullptr;
    if constexpr (LIDS) {
        lids = reinterpret_cast<uint16_t *>(
            pool_lds + (LDS == STATE_GLOBAL ? 0 : size_t(M.n) * lds_stride<LDS>()));
        lds_ids_fill(V, M, kmax, lids);
    }
    if constexpr (LDS != STATE_GLOBAL || LIDS) __syncthreads();
    // step -1 is the initial acceleration pass of a system without valid
    // accelerations; one call site keeps a single copy of the pass in the code
    for (int s = M.acc_valid ? 0 : -1; s < int(nsteps); s++) {
        if (s >= 0) {
            pool_kick_drift<LDS>(V, M, s > 0, half, dt, g0, g_end, gs);
            if (s > 0 && threadIdx.x == 0) advance_facets(F, int(M.nf), dt);
            __syncthreads();
        }
        pool_force_phase<BIN, HAM, PAIRS, PREC, LDS, LIDS, FAC>(P, MC, V, M, cur, F, g0, g_end, gs, lids, kmax);
        cur ^= 1u;
        __syncthreads();
    }
    if (nsteps > 0) {
        pool_final_kick<LDS>(V, M, half, g0, g_end, gs);
        if (threadIdx.x == 0) advance_facets(F, int(M.nf), dt);
    } else if constexpr (LDS == STATE_FULL) {
        // only the initial pass ran: its accelerations go back to global
        for (uint32_t g = M.offset + threadIdx.x; g < M.offset + M.n; g += blockDim.x) {
            const double *q = lds_rec<LDS>(M.offset, g);
            st3(V.a, g, lds3(q + 12));
            st3(V.al, g, lds3(q + 15));
        }
    }
    __syncthreads();
}

// One system's interval by the whole workgroup, in the state tier its size
// allows (s_red: block_max_u32's scratch words).
template <int BIN, int HAM, int PAIRS, int PREC, bool FAC>
__device__ __forceinline__ void run_one(const hg_params &P, const mixed_consts &MC, const pool_view &V,
                                        uint32_t slot, uint32_t nsteps, double dt, uint32_t lds_bytes,
                                        uint32_t *s_red) {
    const pool_meta M = V.meta[slot];
    facet_dev *F = V.facets + size_t(slot) * V.max_facets;
    const size_t need = size_t(M.n) * sizeof(double);
    if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) {
        // the partner ids go to LDS too wherever they fit beside the state
        uint32_t kmax = 0;
        for (uint32_t t = threadIdx.x; t < M.n; t += blockDim.x) kmax = max(kmax, V.ncnt[M.offset + t]);
        kmax = block_max_u32(kmax, s_red);
        const size_t ids = M.n <= 65535u ? lds_ids_bytes(M.n, kmax) : ~size_t(0) / 2;
        if (need * kFullStride + ids <= lds_bytes)
            run_system<BIN, HAM, PAIRS, PREC, STATE_FULL, true, FAC>(P, MC, V, M, F, nsteps, dt, kmax);
        else if (need * kMirrorStride + ids <= lds_bytes)
            run_system<BIN, HAM, PAIRS, PREC, STATE_MIRROR, true, FAC>(P, MC, V, M, F, nsteps, dt, kmax);
        else if (need * kPosStride + ids <= lds_bytes)
            run_system<BIN, HAM, PAIRS, PREC, STATE_POS, true, FAC>(P, MC, V, M, F, nsteps, dt, kmax);
        else if (ids <= lds_bytes)
            run_system<BIN, HAM, PAIRS, PREC, STATE_GLOBAL, true, FAC>(P, MC, V, M, F, nsteps, dt, kmax);
        else
            run_system<BIN, HAM, PAIRS, PREC, STATE_GLOBAL, false, FAC>(P, MC, V, M, F, nsteps, dt, 0);
    } else {
        if (need * kFullStride <= lds_bytes)
            run_system<BIN, HAM, PAIRS, PREC, STATE_FULL, false, FAC>(P, MC, V, M, F, nsteps, dt, 0);
        else if (need * kMirrorStride <= lds_bytes)
            run_system<BIN, HAM, PAIRS, PREC, STATE_MIRROR, false, FAC>(P, MC, V, M, F, nsteps, dt, 0);
        else
            run_system<BIN, HAM, PAIRS, PREC, STATE_GLOBAL, false, FAC>(P, MC, V, M, F, nsteps, dt, 0);
    }
}

// Several small systems (a pack: count members, all of them at most one
// particle per thread together) stepped side by side by one workgroup, so
// that a system of 100 particles does not leave 400 lanes idle through every
// step. Neighbour-list mode, all state in LDS: member m's particles take pack
// positions base_m .. base_m + n_m - 1 (thread = position). Each thread steps
// its own particle with the single-system device code, given its member's
// meta with offset_m - base_m in place of the offset: LDS records and partner
// ids are addressed by (arena index - that offset) = pack position (unsigned
// arithmetic), and the ids are stored as pack positions. Every operation of a
// particle is that of run_system, so a system's result does not depend on
// packing. Returns false, having done nothing, when the pack needs more
// threads or LDS than the workgroup has; the caller then steps the members
// one at a time.
constexpr uint32_t kMaxPack = 8;
template <int BIN, int HAM, int PREC, bool FAC>
__device__ __forceinline__ bool run_pack(const hg_params &P, const mixed_consts &MC, const pool_view &V,
                                         const uint32_t *slots, uint32_t cnt, uint32_t nsteps, double dt,
                                         uint32_t lds_bytes, uint32_t *s_red, pool_meta *s_pm, uint32_t *s_base) {
    if (threadIdx.x == 0) {
        uint32_t base = 0;
        for (uint32_t m = 0; m < cnt; m++) {
            s_pm[m] = V.meta[slots[m]];
            s_base[m] = base;
            base += s_pm[m].n;
        }
        s_base[cnt] = base;
    }
    __syncthreads();
    const uint32_t N = s_base[cnt], t = threadIdx.x;
    uint32_t m = 0;
    bool all_valid = true;
    for (uint32_t k = 0; k < cnt; k++) {
        if (k > 0 && t >= s_base[k]) m = k;
        all_valid = all_valid && s_pm[k].acc_valid;
    }
    const bool own = t < N;
    const pool_meta Pm = s_pm[m];
    const uint32_t g = Pm.offset + (t - s_base[m]);
    pool_meta Mv = Pm;
    Mv.offset = Pm.offset - s_base[m];
    Mv.n = N;
    uint32_t kmax = own ? V.ncnt[g] : 0u;
    kmax = block_max_u32(kmax, s_red);
    if (N > blockDim.x || size_t(N) * sizeof(double) * kFullStride + lds_ids_bytes(N, kmax) > lds_bytes) return false;
    facet_dev *F = V.facets + size_t(Pm.slot) * V.max_facets;
    uint16_t *lids = reinterpret_cast<uint16_t *>(pool_lds + size_t(N) * kFullStride);
    if (own) {
        double *q = pool_lds + size_t(t) * kFullStride;
        sds3(q, ld3(V.x, g));
        sds3(q + 3, ld3(V.v, g));
        sds3(q + 6, ld3(V.w, g));
        sds3(q + 9, ld3(V.th, g));
        sds3(q + 12, ld3(V.a, g));
        sds3(q + 15, ld3(V.al, g));
        const uint32_t c = V.ncnt[g];
        lids[kmax * N + t] = uint16_t(c);
        for (uint32_t k = 0; k < c; k++) lids[k * N + t] = uint16_t(V.nb[size_t(k) * V.stride + g] - Mv.offset);
    }
    __syncthreads();
    const double half = dt / 2.0;
    uint32_t cur = Pm.cur;
    auto advance_all = [&]() {
        for (uint32_t k = 0; k < cnt; k++)
            advance_facets(V.facets + size_t(s_pm[k].slot) * V.max_facets, int(s_pm[k].nf), dt);
    };
    for (int s = all_valid ? 0 : -1; s < int(nsteps); s++) {
        if (s >= 0) {
            if (own) pool_kick_drift<STATE_FULL>(V, Mv, s > 0, half, dt, g, g + 1, 1);
            if (s > 0 && t == 0) advance_all();
            __syncthreads();
        }
        if (own && (s >= 0 || !Pm.acc_valid)) {
            pool_force_phase<BIN, HAM, HG_PAIRS_NEIGHBOR_LIST, PREC, STATE_FULL, true, FAC>(P, MC, V, Mv, cur, F, g,
                                                                                           g + 1, 1, lids, kmax);
            cur ^= 1u;
        }
        __syncthreads();
    }
    if (nsteps > 0) {
        if (own) pool_final_kick<STATE_FULL>(V, Mv, half, g, g + 1, 1);
        if (t == 0) advance_all();
    } else if (own) {
        const double *q = pool_lds + size_t(t) * kFullStride;
        st3(V.a, g, lds3(q + 12));
        st3(V.al, g, lds3(q + 15));
    }
    __syncthreads();
    return true;
}

// One rebuild interval of every queued system. The queue holds packs
// (packs[i] = first | count << 24 over the slots in `order`): a pack of one
// is a system stepped by the whole workgroup, a larger one small systems
// stepped side by side (run_pack). Exit: every workgroup leaves once the
// shared counter passes `count`. lds_bytes of dynamic LDS per workgroup
// decide each system's state placement. FAC = false leaves the facet fold
// out (every queued system has nf = 0): it holds the kernel's largest
// register set. TPB threads per workgroup (256 or 512): a 512-thread
// workgroup alone on a CU has the same waves per SIMD as two of 256 and twice
// the LDS for one system.
template <int BIN, int HAM, int PAIRS, int PREC, bool FAC, int TPB>
// The model constants come by value: the scalar registers they spill to are
// re-read with v_readlane, which measured faster than reloading them through
// a pointer inside the pair loop (scalar loads add memory latency there).
__global__ void __launch_bounds__(TPB, HG_CHUNK_MIN_BLOCKS)
    k_pool_chunk(hg_params P, mixed_consts MC, pool_view V, const uint32_t *order, const uint32_t *packs,
                 uint32_t count, uint32_t *counter, uint32_t nsteps, double dt, uint32_t lds_bytes) {
    __shared__ uint32_t s_item;
    __shared__ uint32_t s_red[TPB / 64];
    __shared__ pool_meta s_pm[kMaxPack];
    __shared__ uint32_t s_base[kMaxPack + 1];
    for (;;) {
        if (threadIdx.x == 0) s_item = atomicAdd(counter, 1u);
        __syncthreads();
        const uint32_t item = s_item;
        __syncthreads();
        if (item >= count) break;
        const uint32_t pk = packs[item];
        const uint32_t first = pk & 0xFFFFFFu, cnt = pk >> 24;
        if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) {
            if (cnt > 1 &&
                run_pack<BIN, HAM, PREC, FAC>(P, MC, V, order + first, cnt, nsteps, dt, lds_bytes, s_red, s_pm, s_base))
                continue;
        }
        for (uint32_t k = 0; k < cnt; k++)
            run_one<BIN, HAM, PAIRS, PREC, FAC>(P, MC, V, order[first + k], nsteps, dt, lds_bytes, s_red);
    }
}

template <int BIN, int HAM, int PREC>
__global__ void __launch_bounds__(kWalkBlock)
    k_walk_force(hg_params P, mixed_consts MC, pool_view V, const wide_block *map, int pass) {
    const wide_block b = map[blockIdx.x];
    const pool_meta M = V.meta[b.slot];
    if (pass < 0 && M.acc_valid) return;
    const uint32_t passed = pass < 0 ? 0u : uint32_t(pass) + (M.acc_valid ? 0u : 1u);
    const uint32_t g = M.offset + b.start + threadIdx.x;
    if (g >= M.offset + M.n) return;
    pool_force_phase<BIN, HAM, HG_PAIRS_ALL, PREC, STATE_GLOBAL>(
        P, MC, V, M, M.cur ^ (passed & 1u), V.facets + size_t(b.slot) * V.max_facets, g, g + 1, 1);
}

}  // namespace
}  // namespace hg

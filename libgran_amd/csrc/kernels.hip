// gfx950 kernels of the FP64 DEM step: acceleration pass (pair fold + facets),
// velocity-Verlet kick/drift, cell-list neighbour rebuild and diagnostics.
//
// Data layout in HBM
//   particle fields x, v, theta, omega, a, alpha: one array per field, 4
//     doubles (32 B) per particle, so a particle's vector is one aligned
//     32-byte load and a wavefront's loads are contiguous.
//   neighbour list: transposed fixed-capacity slots, nb[k*n + i], ascending j
//     per particle; consecutive lanes (particles) read consecutive words.
//   pair-state table: per particle a j-sorted list of (tag, spring9) where
//     tag = j | bonded-bit; tags transposed as pj[s*n + i], springs in one
//     contiguous 80-byte record per entry at ps[(s*n + i)*10].
//     It holds every bonded pair and every pair whose contact spring the
//     reference would hold non-zero. Each acceleration pass reads the old
//     table and writes the new one while walking the partners in ascending j,
//     so spring state survives neighbour rebuilds with no separate merge.
#include <hip/hip_runtime.h>

#include "hg_internal.h"
#include "pair_eval.h"

namespace hg {

namespace {


// Neighbour-list acceleration pass: one lane per particle i, partners in the
// list's ascending order, so the per-particle sum has the reference's order.
// TRACK: the particle's share of its pairs' dissipated work this step is
// added to S.diss (4 doubles per particle: normal, tangential, rolling,
// torsion).
template <int BIN, int HAM, bool TRACK = false>
__device__ __forceinline__ void force_nl_one(const hg_params &P, const sys_view &S, uint32_t i) {
    const d3 xi = ld3(S.x, i), vi = ld3(S.v, i), wi = ld3(S.w, i);
    acc6 acc{zero3(), zero3()};
    walker_t<false> W;
    if constexpr (BIN != HG_BINARY_NONE) W.init(S.pt, i);
    if constexpr (BIN == HG_BINARY_SINTER_LEGACY) W.init_legacy(S.pt);
    id_list ids;
    ids.init(S.nb, S.ncnt, S.n, i, S.cap_n);
    double d4[4] = {0.0, 0.0, 0.0, 0.0};
    nl_partners(ids, [&](uint32_t j) { return pstate{ld3(S.x, j), ld3(S.v, j), ld3(S.w, j)}; },
                [&](uint32_t j, const pstate &sj) {
                    pair_fold_vw<BIN, HAM, TRACK>(P, j, xi, vi, wi, sj.x, [&](d3 &v, d3 &w) { v = sj.v, w = sj.w; },
                                                  W, acc, d4);
                });
    close_table<BIN>(W, S.pt.pcnt_new, i, S.flags);
    if (S.nf > 0) acc = acc + facet_fold(P, S.facets, S.nf, S.ss, S.n, i, xi, vi, wi);
    st3(S.a, i, acc.lin);
    st3(S.al, i, acc.ang);
    if constexpr (TRACK)
        for (int c = 0; c < 4; c++) S.diss[4 * size_t(i) + c] = S.diss[4 * size_t(i) + c] + d4[c];
}

template <int BIN, int HAM, bool TRACK>
__global__ void __launch_bounds__(256) k_force_nl(hg_params P, sys_view S) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.n) return;
    force_nl_one<BIN, HAM, TRACK>(P, S, i);
}

// All-pairs acceleration pass (granular_system): every j != i in ascending
// order. Partner state is staged through LDS one tile per block-wide step;
// all lanes read the same LDS word, a broadcast with no bank conflict.
constexpr int kTile = 256;
struct tile_lds {
    double sx[3][kTile], sv[3][kTile], sw[3][kTile];
};
// The pass for particle i = blockIdx.x * blockDim.x + threadIdx.x; every
// thread of the block takes part (it stages tiles), live or not.
template <int BIN, int HAM, bool TRACK = false>
__device__ __forceinline__ void force_all_block(const hg_params &P, const sys_view &S, tile_lds &T) {
    auto &sx = T.sx;
    auto &sv = T.sv;
    auto &sw = T.sw;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < S.n;
    d3 xi = zero3(), vi = zero3(), wi = zero3();
    if (live) {
        xi = ld3(S.x, i);
        vi = ld3(S.v, i);
        wi = ld3(S.w, i);
    }
    acc6 acc{zero3(), zero3()};
    double d4[4] = {0.0, 0.0, 0.0, 0.0};
    walker_t<false> W;
    if constexpr (BIN != HG_BINARY_NONE) {
        if (live) W.init(S.pt, i);
    }
    if constexpr (BIN == HG_BINARY_SINTER_LEGACY) {
        if (live) W.init_legacy(S.pt);
    }
    for (uint32_t base = 0; base < S.n; base += kTile) {
        __syncthreads();
        for (uint32_t t = threadIdx.x; t < kTile && base + t < S.n; t += blockDim.x) {
            d3 q = ld3(S.x, base + t), u = ld3(S.v, base + t), r = ld3(S.w, base + t);
            sx[0][t] = q.x; sx[1][t] = q.y; sx[2][t] = q.z;
            sv[0][t] = u.x; sv[1][t] = u.y; sv[2][t] = u.z;
            sw[0][t] = r.x; sw[1][t] = r.y; sw[2][t] = r.z;
        }
        __syncthreads();
        if (live) {
            const uint32_t m = (S.n - base) < uint32_t(kTile) ? (S.n - base) : uint32_t(kTile);
            for (uint32_t jj = 0; jj < m; jj++) {
                const uint32_t j = base + jj;
                if (j == i) continue;
                pair_fold_vw<BIN, HAM, TRACK>(
                    P, j, xi, vi, wi, d3{sx[0][jj], sx[1][jj], sx[2][jj]},
                    [&](d3 &v, d3 &w) { v = d3{sv[0][jj], sv[1][jj], sv[2][jj]}, w = d3{sw[0][jj], sw[1][jj], sw[2][jj]}; },
                    W, acc, d4);
            }
        }
    }
    if (!live) return;
    close_table<BIN>(W, S.pt.pcnt_new, i, S.flags);
    if (S.nf > 0) acc = acc + facet_fold(P, S.facets, S.nf, S.ss, S.n, i, xi, vi, wi);
    st3(S.a, i, acc.lin);
    st3(S.al, i, acc.ang);
    if constexpr (TRACK)
        for (int c = 0; c < 4; c++) S.diss[4 * size_t(i) + c] = S.diss[4 * size_t(i) + c] + d4[c];
}

template <int BIN, int HAM, bool TRACK>
__global__ void __launch_bounds__(kTile) k_force_all(hg_params P, sys_view S) {
    __shared__ tile_lds T;
    force_all_block<BIN, HAM, TRACK>(P, S, T);
}

// Kick (completing the previous step when `pending`), kick, drift:
//   v += a*(dt/2); w += alpha*(dt/2); x += v*dt; theta += w*dt.
// Lane 0 of block 0 advances the facets when a previous step completes here.
__device__ __forceinline__ void kick_drift_one(double *x, double *v, double *th, double *w, const double *a,
                                               const double *al, uint32_t i, int pending, double half_prev,
                                               double half, double dt) {
    d3 vi = ld3(v, i), wi = ld3(w, i);
    const d3 ai = ld3(a, i), ali = ld3(al, i);
    if (pending) {
        vi = vi + ai * half_prev;
        wi = wi + ali * half_prev;
    }
    vi = vi + ai * half;
    wi = wi + ali * half;
    st3(x, i, ld3(x, i) + vi * dt);
    st3(th, i, ld3(th, i) + wi * dt);
    st3(v, i, vi);
    st3(w, i, wi);
}

__global__ void __launch_bounds__(256) k_kick_drift(double *x, double *v, double *th, double *w, const double *a,
                                                    const double *al, uint32_t n, int pending, double half_prev,
                                                    double half, double dt, facet_dev *facets, int nf,
                                                    double facet_dt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (pending && i == 0) advance_facets(facets, nf, facet_dt);
    if (i >= n) return;
    kick_drift_one(x, v, th, w, a, al, i, pending, half_prev, half, dt);
}

// sinter_step_handler (sinter_bridge.h:24-42, 55-75) after a drift: each of
// particle i's connectors moves by dx = v_i dt (increment_x), then turns by
// dtheta = w_i dt about the new centre (increment_theta). v, w and x are the
// values the drift just used and wrote, so dx and dtheta are its increments.
__device__ __forceinline__ void legacy_move_one(const double *x, const double *v, const double *w, uint32_t n,
                                                uint32_t i, double dt, double *lconn, const uint32_t *bcnt) {
    const d3 dx = ld3(v, i) * dt, dth = ld3(w, i) * dt, xi = ld3(x, i);
    const uint32_t c = bcnt[i];
    for (uint32_t s = 0; s < c; s++) {
        double *r = lconn + (size_t(s) * n + i) * kConnRec;
        for (int q = 0; q < 5; q++) {
            d3 p = d3{r[3 * q], r[3 * q + 1], r[3 * q + 2]} + dx;
            const d3 spring_vector = p - xi;
            p = p + cross(dth, spring_vector);
            r[3 * q] = p.x;
            r[3 * q + 1] = p.y;
            r[3 * q + 2] = p.z;
        }
    }
}

__global__ void __launch_bounds__(256) k_legacy_move(const double *x, const double *v, const double *w, uint32_t n,
                                                     double dt, double *lconn, const uint32_t *bcnt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    legacy_move_one(x, v, w, n, i, dt, lconn, bcnt);
}

// Closing kick of particle i; a non-finite result raises FLAG_NUMERIC.
__device__ __forceinline__ void final_kick_one(double *v, double *w, const double *a, const double *al, uint32_t i,
                                               double half, int *flags) {
    const d3 vi = ld3(v, i) + ld3(a, i) * half, wi = ld3(w, i) + ld3(al, i) * half;
    st3(v, i, vi);
    st3(w, i, wi);
    if (nonfinite(vi, wi)) atomicOr(&flags[FLAG_NUMERIC], 1);
}

__global__ void __launch_bounds__(256) k_final_kick(double *v, double *w, const double *a, const double *al,
                                                    uint32_t n, double half, facet_dev *facets, int nf,
                                                    double facet_dt, int *flags) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) advance_facets(facets, nf, facet_dt);
    if (i >= n) return;
    final_kick_one(v, w, a, al, i, half, flags);
}

// nsteps steps of a legacy sinter_functor system of at most kTile particles in
// one workgroup, one particle per thread: per step the kick/drift (with the
// legacy connector moves), a barrier, the acceleration pass, a barrier, and at
// the end the closing kick, as the per-step launches of k_kick_drift,
// k_legacy_move, k_force_nl / k_force_all and k_final_kick do it, through the
// same device code. The pass reads pair-state table `even` on even steps and
// `odd` on odd ones (the two halves swap every pass).
template <int BIN, int HAM>
__global__ void __launch_bounds__(kTile) k_small_steps(hg_params P, sys_view even, sys_view odd, double *x, double *v,
                                                       double *th, double *w, facet_dev *facets, uint32_t nsteps,
                                                       double half, double dt, int nf_advance, double *lconn,
                                                       const uint32_t *bcnt) {
    __shared__ tile_lds T;
    const uint32_t i = threadIdx.x;
    const uint32_t n = even.n;
    const bool live = i < n;
    for (uint32_t s = 0; s < nsteps; s++) {
        const bool pending = s > 0;
        if (pending && i == 0) advance_facets(facets, nf_advance, dt);
        if (live) {
            kick_drift_one(x, v, th, w, even.a, even.al, i, pending, half, half, dt);
            if (lconn) legacy_move_one(x, v, w, n, i, dt, lconn, bcnt);
        }
        __syncthreads();
        if (P.pair_mode == HG_PAIRS_NEIGHBOR_LIST) {
            if (live) force_nl_one<BIN, HAM>(P, (s & 1u) ? odd : even, i);
        } else {
            force_all_block<BIN, HAM>(P, (s & 1u) ? odd : even, T);
        }
        __syncthreads();
    }
    if (i == 0) advance_facets(facets, nf_advance, dt);
    if (live) final_kick_one(v, w, even.a, even.al, i, half, even.flags);
}

// triangular_facet::update_positions with the driver's velocity (one lane).
__global__ void k_advance_facet(facet_dev *f, double vx, double vy, double vz, double dt) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        f->v_facet = d3{vx, vy, vz};
        for (int k = 0; k < 3; k++) f->vert[k] = f->vert[k] + f->v_facet * dt;
    }
}

__global__ void k_zero_u32(uint32_t *p, size_t count) {
    for (size_t k = blockIdx.x * size_t(blockDim.x) + threadIdx.x; k < count; k += size_t(gridDim.x) * blockDim.x)
        p[k] = 0;
}
__global__ void k_zero_f64(double *p, size_t count) {
    for (size_t k = blockIdx.x * size_t(blockDim.x) + threadIdx.x; k < count; k += size_t(gridDim.x) * blockDim.x)
        p[k] = 0.0;
}

__global__ void __launch_bounds__(64) k_copy_words(const int *src, int *dst, int count) {
    for (int k = int(threadIdx.x); k < count; k += 64) dst[k] = src[k];
}

// Bound by the link to the host: consecutive lanes write consecutive words.
struct pack_src {
    const double *f[4];
};
__global__ void __launch_bounds__(256) k_pack3(pack_src F, size_t words, double *out) {
    const double *src = F.f[blockIdx.y];
    for (size_t q = blockIdx.x * size_t(blockDim.x) + threadIdx.x; q < words; q += size_t(gridDim.x) * blockDim.x)
        out[blockIdx.y * words + q] = src[q / 3 * 4 + q % 3];
}

// ---------------------------------------------------- neighbour rebuild -----
// Exclusive scan in three launches: per-block scan of kScanChunk words with
// block totals, a single-block scan of the totals, then the offsets added.
constexpr uint32_t kScanThreads = 256, kScanPer = 8, kScanChunk = kScanThreads * kScanPer;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *sh, uint32_t &total) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t off = 1; off < blockDim.x; off <<= 1) {
        uint32_t add = threadIdx.x >= off ? sh[threadIdx.x - off] : 0u;
        __syncthreads();
        sh[threadIdx.x] += add;
        __syncthreads();
    }
    total = sh[blockDim.x - 1];
    uint32_t r = sh[threadIdx.x] - v;
    __syncthreads();
    return r;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_blocks(const uint32_t *in, uint32_t *out, uint32_t count,
                                                               uint32_t *block_sums) {
    __shared__ uint32_t sh[kScanThreads];
    const uint32_t base = blockIdx.x * kScanChunk + threadIdx.x * kScanPer;
    uint32_t vals[kScanPer];
    uint32_t s = 0;
    for (uint32_t k = 0; k < kScanPer; k++) {
        vals[k] = base + k < count ? in[base + k] : 0u;
        s += vals[k];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan(s, sh, total);
    for (uint32_t k = 0; k < kScanPer; k++) {
        if (base + k < count) out[base + k] = run;
        run += vals[k];
    }
    if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_top(uint32_t *block_sums, uint32_t nblocks) {
    __shared__ uint32_t sh[kScanThreads];
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nblocks; base += kScanThreads) {
        const uint32_t idx = base + threadIdx.x;
        const uint32_t v = idx < nblocks ? block_sums[idx] : 0u;
        uint32_t total;
        const uint32_t r = block_exclusive_scan(v, sh, total);
        if (idx < nblocks) block_sums[idx] = r + carry;
        carry += total;
    }
}

__global__ void __launch_bounds__(kScanThreads) k_scan_add(uint32_t *out, uint32_t count, const uint32_t *block_sums) {
    const uint32_t add = block_sums[blockIdx.x];
    const uint32_t base = blockIdx.x * kScanChunk;
    for (uint32_t k = threadIdx.x; k < kScanChunk && base + k < count; k += blockDim.x) out[base + k] += add;
}

__device__ __forceinline__ uint32_t cell_hash(uint32_t slot, long long cx, long long cy, long long cz, uint32_t mask) {
    uint64_t h = uint64_t(cx) * 73856093ull ^ uint64_t(cy) * 19349663ull ^ uint64_t(cz) * 83492791ull ^
                 uint64_t(slot) * 2654435761ull;
    h ^= h >> 29;
    h *= 0xbf58476d1ce4e5b9ull;
    h ^= h >> 32;
    return uint32_t(h) & mask;
}

__device__ __forceinline__ void cell_coords(d3 q, double cs, long long &cx, long long &cy, long long &cz) {
    cx = (long long)floor(q.x / cs);
    cy = (long long)floor(q.y / cs);
    cz = (long long)floor(q.z / cs);
}

__global__ void __launch_bounds__(256) k_cell_count(list_build B, double cs) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= B.count) return;
    const uint32_t slot = B.owner ? B.owner[g] : 0u;
    if (slot == kNoEntry || (B.meta && !B.meta[slot].rebuild)) {
        B.cell_of[g] = kNoEntry;
        return;
    }
    long long cx, cy, cz;
    cell_coords(ld3(B.x, g), cs, cx, cy, cz);
    const uint32_t h = cell_hash(slot, cx, cy, cz, B.hash_size - 1);
    B.cell_of[g] = h;
    atomicAdd(&B.buckets[h], 1u);
}

__global__ void __launch_bounds__(256) k_cell_fill(list_build B) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= B.count) return;
    const uint32_t h = B.cell_of[g];
    if (h == kNoEntry) return;
    const d3 p = ld3(B.x, g);
    B.recs[B.bucket_start[h] + atomicAdd(&B.buckets[B.hash_size + h], 1u)] =
        cell_rec{p.x, p.y, p.z, g, B.owner ? B.owner[g] : 0u};
}

// The reference predicate norm(x_i - x_j) < r_verlet behind a squared-distance
// prefilter: a correctly rounded sqrt(d2) < r_verlet implies d2 < r_verlet^2
// (1 + 2^-52), so this bound drops no pair the exact test keeps; squares below
// the smallest normal number have few bits and go to the exact test.
struct in_range {
    double r, d2_max;
    __device__ __forceinline__ in_range(double r_verlet)
        : r(r_verlet), d2_max(fmax(r_verlet * r_verlet * (1.0 + 1e-12), 0x1p-1022)) {}
    __device__ __forceinline__ bool operator()(d3 d) const { return dot(d, d) < d2_max && norm(d) < r; }
};

__device__ __forceinline__ void close_list(const list_build &B, uint32_t g, uint32_t slot, uint32_t cnt) {
    B.ncnt[g] = cnt < B.cap ? cnt : B.cap;
    if (cnt > B.cap) {
        atomicOr(&B.flags[FLAG_NL_OVERFLOW], 1);
        atomicMax(&B.flags[FLAG_NL_MAXCOUNT], int(cnt));
        if (B.sflags) atomicOr(&B.sflags[slot], HG_FAULT_NEIGHBOR_CAPACITY);
    }
}

// Lists from the cell records, eight lanes a particle. Cells are twice the
// list radius wide, so a partner lies in the particle's own cell or the
// neighbour on the side of the half the particle sits in, along each axis: 2 x
// 2 x 2 cells, one for each lane. (In cell units a partner is less than 0.5 (1
// - 1e-9) away; a particle in the lower half, u - floor(u) < 0.5, has its
// partners in floor(u) - 1 .. floor(u), one in the upper half in floor(u) ..
// floor(u) + 1. That holds however far out the system lies: u is one correctly
// rounded quotient, and rounding cannot carry a value past a whole or a half,
// so a particle that the rounding moves to the upper half, from within half a
// unit in the last place below it, has its partners at floor(u) or above after
// rounding too. Cells laid from one of the particles, u = (x - o) / cs, round
// twice, and where that particle is far away from the others pairs were
// missed.) The matches go to LDS and from there to their rank among
// them, so the list ascends. One lane walking all eight buckets took 104 us at
// 20,000 particles, each bucket a chain of dependent reads.
constexpr uint32_t kListLanes = 8, kListParts = 256 / kListLanes, kListMost = 96, kRecBatch = 4;
__global__ void __launch_bounds__(256) k_list_fill(list_build B, double cs) {
    __shared__ uint32_t s_cnt[kListParts];
    __shared__ uint32_t s_list[kListParts][kListMost];
    const uint32_t lane = threadIdx.x % kListLanes, p = threadIdx.x / kListLanes;
    const uint32_t g = blockIdx.x * kListParts + p;
    const bool on = g < B.count && B.cell_of[g] != kNoEntry;
    if (lane == 0) s_cnt[p] = 0;
    __syncthreads();
    const uint32_t slot = on && B.owner ? B.owner[g] : 0u;
    const d3 xi = on ? ld3(B.x, g) : zero3();
    const in_range near(B.r_verlet);
    long long bx, by, bz;
    cell_coords(xi, cs, bx, by, bz);
    bx -= xi.x / cs - double(bx) < 0.5 ? 1 : 0;
    by -= xi.y / cs - double(by) < 0.5 ? 1 : 0;
    bz -= xi.z / cs - double(bz) < 0.5 ? 1 : 0;
    // calls match(j) for every partner in the bucket of cell c of the eight
    auto scan = [&](uint32_t h, auto &&match) {
        const uint32_t b = B.bucket_start[h], e = b + B.buckets[h];
        for (uint32_t q = b; q < e; q += kRecBatch) {
            // records loaded together (the last one again past the end) overlap
            cell_rec c[kRecBatch];
#pragma unroll
            for (uint32_t k = 0; k < kRecBatch; k++) c[k] = B.recs[q + k < e ? q + k : e - 1];
#pragma unroll
            for (uint32_t k = 0; k < kRecBatch; k++)
                if (q + k < e && c[k].j != g && c[k].slot == slot && near(xi - d3{c[k].x, c[k].y, c[k].z}))
                    match(c[k].j);
        }
    };
    auto hash_of = [&](uint32_t c) {
        return cell_hash(slot, bx + (c & 1), by + (c >> 1 & 1), bz + (c >> 2), B.hash_size - 1);
    };
    const uint32_t h = hash_of(lane);
    bool dup = false;  // a bucket shared by two of the cells is scanned once
    for (uint32_t c = 0; c < kListLanes - 1; c++) {
        const uint32_t hc = uint32_t(__shfl(int(h), int(c), int(kListLanes)));
        dup |= c < lane && hc == h;
    }
    if (on && !dup)
        scan(h, [&](uint32_t j) {
            const uint32_t at = atomicAdd(&s_cnt[p], 1u);
            if (at < kListMost) s_list[p][at] = j;
        });
    __syncthreads();
    if (!on) return;
    const uint32_t cnt = s_cnt[p];
    if (cnt <= kListMost) {
        for (uint32_t e = lane; e < cnt; e += kListLanes) {
            const uint32_t j = s_list[p][e];
            uint32_t rank = 0;
            for (uint32_t f = 0; f < cnt; f++) rank += s_list[p][f] < j ? 1u : 0u;
            if (rank < B.cap) B.nb[size_t(rank) * B.stride + g] = j;
        }
    } else if (lane == 0) {
        // a list longer than the LDS row: by insertion, one lane
        uint32_t n = 0;
        for (uint32_t c = 0; c < kListLanes; c++) {
            const uint32_t hc = hash_of(c);
            bool seen = false;
            for (uint32_t q = 0; q < c; q++) seen |= hash_of(q) == hc;
            if (seen) continue;
            scan(hc, [&](uint32_t j) {
                uint32_t pos = n < B.cap ? n : B.cap;
                if (pos == B.cap) {  // full: j displaces the largest kept one, or is dropped
                    if (B.cap == 0 || B.nb[size_t(B.cap - 1) * B.stride + g] < j) {
                        n++;
                        return;
                    }
                    pos--;
                }
                while (pos > 0 && B.nb[size_t(pos - 1) * B.stride + g] > j) {
                    B.nb[size_t(pos) * B.stride + g] = B.nb[size_t(pos - 1) * B.stride + g];
                    pos--;
                }
                B.nb[size_t(pos) * B.stride + g] = j;
                n++;
            });
        }
    }
    if (lane == 0) close_list(B, g, slot, cnt);
}

// Every pair tested: one launch instead of the cell list's seven, whose
// latency a small system pays in full. A wavefront lists four particles, 64
// candidates at a time from LDS; the ballot gives each match its place, in
// ascending order. Work grows with n^2 and is hidden behind the cell list's
// launches up to kBruteListMax.
constexpr uint32_t kBruteEach = 4, kBruteParts = 4 * kBruteEach;
__global__ void __launch_bounds__(256) k_list_brute(list_build B) {
    __shared__ double sx[3][256];
    const uint32_t lane = threadIdx.x & 63u, first = blockIdx.x * kBruteParts + (threadIdx.x >> 6) * kBruteEach;
    const in_range near(B.r_verlet);
    d3 xi[kBruteEach];
    uint32_t cnt[kBruteEach];
#pragma unroll
    for (uint32_t q = 0; q < kBruteEach; q++) {
        xi[q] = first + q < B.count ? ld3(B.x, first + q) : zero3();
        cnt[q] = 0;
    }
    for (uint32_t base = 0; base < B.count; base += 256) {
        __syncthreads();
        if (base + threadIdx.x < B.count) {
            const d3 a = ld3(B.x, base + threadIdx.x);
            sx[0][threadIdx.x] = a.x;
            sx[1][threadIdx.x] = a.y;
            sx[2][threadIdx.x] = a.z;
        }
        __syncthreads();
        for (uint32_t t = lane; t < 256u && base + t - lane < B.count; t += 64) {
            const uint32_t j = base + t;
            const bool live = j < B.count;
            const d3 xj = live ? d3{sx[0][t], sx[1][t], sx[2][t]} : zero3();
#pragma unroll
            for (uint32_t q = 0; q < kBruteEach; q++) {
                const uint32_t i = first + q;
                const bool hit = live && i < B.count && j != i && near(xi[q] - xj);
                const uint64_t m = __ballot(hit);
                if (hit) {
                    const uint32_t at = cnt[q] + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
                    if (at < B.cap) B.nb[size_t(at) * B.stride + i] = j;
                }
                cnt[q] += uint32_t(__popcll(m));
            }
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < kBruteEach; q++)
        if (lane == 0 && first + q < B.count) close_list(B, first + q, 0, cnt[q]);
}

// ---------------------------------------------------------- diagnostics -----
// Single block: out = KE_total, KE_trans, KE_rot, |P|, |L|, Rg, cm(3).
__global__ void __launch_bounds__(1024) k_diag(const double *x, const double *v, const double *w, uint32_t n,
                                               double mass, double inertia, double *out) {
    __shared__ double red[8][1024];
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // 2*KE_trans, 2*KE_rot, sum v (3), L (3)
    d3 cmsum = zero3();
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        d3 vi = ld3(v, i), wi = ld3(w, i), xi = ld3(x, i);
        cmsum = cmsum + xi;
        acc[0] += mass * dot(vi, vi);
        acc[1] += inertia * dot(wi, wi);
        acc[2] += vi.x; acc[3] += vi.y; acc[4] += vi.z;
        d3 L = inertia * wi + cross(xi, mass * vi);
        acc[5] += L.x; acc[6] += L.y; acc[7] += L.z;
    }
    for (int c = 0; c < 8; c++) red[c][threadIdx.x] = acc[c];
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int c = 0; c < 8; c++) red[c][threadIdx.x] += red[c][threadIdx.x + s];
        __syncthreads();
    }
    __syncthreads();
    double k0 = red[0][0], k1 = red[1][0];
    d3 P{red[2][0], red[3][0], red[4][0]}, L{red[5][0], red[6][0], red[7][0]};
    __syncthreads();
    red[0][threadIdx.x] = cmsum.x; red[1][threadIdx.x] = cmsum.y; red[2][threadIdx.x] = cmsum.z;
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int c = 0; c < 3; c++) red[c][threadIdx.x] += red[c][threadIdx.x + s];
        __syncthreads();
    }
    const d3 cm = d3{red[0][0], red[1][0], red[2][0]} / double(n);
    __syncthreads();
    double rg = 0.0;
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
        d3 dd = ld3(x, i) - cm;
        rg += dot(dd, dd);
    }
    red[0][threadIdx.x] = rg;
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[0][threadIdx.x] += red[0][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = k0 / 2.0 + k1 / 2.0;
        out[1] = k0 / 2.0;
        out[2] = k1 / 2.0;
        out[3] = mass * norm(P);
        out[4] = norm(L);
        out[5] = sqrt(red[0][0] / double(n));
        out[6] = cm.x;
        out[7] = cm.y;
        out[8] = cm.z;
    }
}

// Energy ledger terms of one particle (see launch_energy). Pair terms are
// split evenly between the two particles of a pair and each ordered pair's
// springs carry half of that pair's spring energy, so the sums over all
// particles count every pair once.
//
// Eight lanes share a particle: each takes every eighth row entry and partner,
// and the eight contributions are added in the order of one lane walking them,
// so the sums do not depend on the split. One lane per particle left 79
// wavefronts at 5,000 particles, each a chain of 13 dependent partners.
__global__ void __launch_bounds__(256) k_energy(hg_params P, energy_view E, double mass, double inertia,
                                                double *out) {
    constexpr uint32_t G = 8;
    const uint32_t k = (blockIdx.x * blockDim.x + threadIdx.x) / G, l = threadIdx.x % G;
    if (k >= E.n) return;
    const uint32_t g = E.offset + k;
    const d3 xi = ld3(E.x, g), vi = ld3(E.v, g), wi = ld3(E.w, g);
    double e[8] = {0.5 * mass * dot(vi, vi), 0.5 * inertia * dot(wi, wi), 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto add = [&](double &to, double term) {
#pragma unroll
        for (uint32_t q = 0; q < G; q++) to += __shfl(term, int(q), int(G));
    };
    const uint32_t cnt = E.pcnt ? E.pcnt[g] : 0u;
    for (uint32_t s0 = 0; s0 < cnt; s0 += G) {
        const uint32_t s = s0 + l;
        double t[3] = {0.0, 0.0, 0.0};
        if (s < cnt) {
            const bool bonded = (E.pj[size_t(s) * E.stride + g] & kBondBit) != 0;
            const spring9 sp = ld_rec(E.ps + (size_t(s) * E.stride + g) * kSpringRec);
            const double kt = bonded ? P.sinter.k_t : P.contact.k_t, kr = bonded ? P.sinter.k_r : P.contact.k_r,
                         ko = bonded ? P.sinter.k_o : P.contact.k_o;
            t[0] = 0.25 * kt * dot(sp.s[0], sp.s[0]);
            t[1] = 0.25 * kr * dot(sp.s[1], sp.s[1]);
            t[2] = 0.25 * ko * dot(sp.s[2], sp.s[2]);
        }
        for (int c = 0; c < 3; c++) add(e[3 + c], t[c]);
    }
    // a partner's share of the bond energies in row order, and of the Hamaker
    // potential; a legacy bond adds five of the first kind
    auto pair = [&](uint32_t j, double (&bond)[5], double &ham) {
        const double dist = norm(xi - ld3(E.x, j));
        uint32_t ls = kNoEntry;
        if (E.lconn)
            for (uint32_t s = 0; s < E.bcnt[g]; s++)
                if (E.bj[size_t(s) * E.stride + g] == j) ls = s;
        if (ls != kNoEntry) {
            // the bond's five connector springs, k_d/2 (|s| - L0)^2 each, half
            // to each ordered pair
            const double *ri = E.lconn + (size_t(ls) * E.stride + g) * kConnRec;
            const double *rj = E.lconn + (size_t(E.lslot[size_t(ls) * E.stride + g]) * E.stride + j) * kConnRec;
            for (int q = 0; q < 5; q++) {
                const d3 sq = d3{rj[3 * q], rj[3 * q + 1], rj[3 * q + 2]} - d3{ri[3 * q], ri[3 * q + 1], ri[3 * q + 2]};
                const double d = (q < 4 ? 2.0 * P.contact.r_part : 0.0) - norm(sq);
                bond[q] = 0.25 * P.sinter.k * d * d;
            }
        } else if (P.binary_model != HG_BINARY_NONE) {
            bool bonded = false;
            for (uint32_t s = 0; s < cnt; s++) {
                const uint32_t tag = E.pj[size_t(s) * E.stride + g];
                if ((tag & kIdxMask) == j) bonded = (tag & kBondBit) != 0;
            }
            if (bonded) {
                const double ov = 2.0 * P.sinter.r_part - dist;
                bond[0] = 0.25 * P.sinter.k * ov * ov;
            } else {
                const double ov = 2.0 * P.contact.r_part - dist;
                if (ov > 0.0) bond[0] = 0.25 * P.contact.k * ov * ov;
            }
        }
        if (P.hamaker_model != HG_HAMAKER_NONE) ham = 0.5 * hamaker_potential(P.hamaker_model, P.hamaker, dist);
    };
    const uint32_t m = E.nb ? E.ncnt[g] : E.n;
    for (uint32_t q0 = 0; q0 < m; q0 += G) {
        const uint32_t q = q0 + l;
        double bond[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, ham = 0.0;
        if (q < m) {
            const uint32_t j = E.nb ? E.nb[size_t(q) * E.stride + g] : E.offset + q;
            if (j != g) pair(j, bond, ham);
        }
        if (E.lconn) {
            for (uint32_t t = 0; t < G; t++)
                for (int c = 0; c < 5; c++) e[2] += __shfl(bond[c], int(t), int(G));
        } else {
            add(e[2], bond[0]);
        }
        add(e[6], ham);
    }
    if (l == 0)
        for (int c = 0; c < 8; c++) out[8 * size_t(k) + c] = e[c];
}

inline unsigned blocks_for(size_t n, unsigned bs) { return unsigned((n + bs - 1) / bs); }

template <int BIN, int HAM, bool TRACK>
hipError_t launch_force_t(const hg_params &p, const sys_view &sv, hipStream_t s) {
    if (sv.n == 0) return hipSuccess;
    if (p.pair_mode != HG_PAIRS_NEIGHBOR_LIST) {
        k_force_all<BIN, HAM, TRACK><<<blocks_for(sv.n, kTile), kTile, 0, s>>>(p, sv);
    } else if constexpr (TRACK || BIN == HG_BINARY_SINTER_LEGACY) {
        // 64-lane blocks spread a modest particle count over more CUs.
        k_force_nl<BIN, HAM, TRACK><<<blocks_for(sv.n, 64), 64, 0, s>>>(p, sv);
    } else {
        return hipErrorInvalidValue;  // tiles
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_force(const hg_params &p, const sys_view &sv, hipStream_t s) {
#define HG_CASE(B, H, TRACK)                                                                        \
    if (p.binary_model == B && p.hamaker_model == H && p.precision == HG_PRECISION_FP64 &&          \
        (sv.diss != nullptr) == TRACK)                                                              \
        return launch_force_t<B, H, TRACK>(p, sv, s);
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_NONE, true)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_FULL, true)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_LIMITED, true)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_SIMPLIFIED, true)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_NONE, true)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_FULL, true)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_LIMITED, true)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_SIMPLIFIED, true)
#define HG_CASES(B)                        \
    HG_CASE(B, HG_HAMAKER_NONE, false)     \
    HG_CASE(B, HG_HAMAKER_FULL, false)     \
    HG_CASE(B, HG_HAMAKER_LIMITED, false)  \
    HG_CASE(B, HG_HAMAKER_SIMPLIFIED, false)
    HG_CASES(HG_BINARY_NONE)
    HG_CASES(HG_BINARY_CONTACT)
    HG_CASES(HG_BINARY_SINTER)
    HG_CASES(HG_BINARY_SINTER_LEGACY)
#undef HG_CASES
#undef HG_CASE
    return hipErrorInvalidValue;
}

// ------------------------------------------------------- tiny systems -----
// All steps between two list rebuilds of a system of a few dozen particles, by
// one workgroup, with everything a step touches in LDS: state, the springs and
// terms of every evaluated ordered pair, connectors, facets. Pair (i, k-th
// partner) has the place i * row + k. A step is three phases: which unbonded
// pairs touch; every pair's term; each particle's sum, kick and drift.
//
// What bounds a step is the longest chain of dependent arithmetic, so a pair
// with springs (bonded or touching) is evaluated by four lanes: three for its
// tangential, rolling and torsion springs, one for its Hamaker term, joined by
// quad permutes; lane c < 3 then finishes component c. In the last phase a
// thread owns one component of one particle. The expressions and their order
// are those of sinter_eval, contact_eval and the per-particle walk.
//
// Measured against one thread per pair with state, rows and springs in global
// memory: 19 particles, contact and Hamaker, list rebuilt every 20 steps 20.2
// -> 5.6 us a step, all pairs 15.2 -> 5.6; the legacy 27-particle lattice 18.8
// -> 4.9.
constexpr uint32_t kTinyThreads = 512;

// Doubles (then words) of LDS a system of n particles needs; maxb: the most
// legacy bonds a particle has (0 without the legacy functor).
struct tiny_layout {
    uint32_t n, row, places, maxb;
    __host__ __device__ tiny_layout(uint32_t n_, uint32_t maxb_)
        : n(n_), row((n_ > 1 ? n_ - 1 : 1) | 1u), places(n_ * ((n_ > 1 ? n_ - 1 : 1) | 1u)), maxb(maxb_) {}
    // state (x, v, omega, theta, a, alpha), terms, springs, facet terms, connectors
    __host__ __device__ size_t doubles() const {
        return size_t(18) * n + size_t(15) * places + size_t(6) * n + size_t(15) * maxb * n;
    }
    // entries, bonded list, touching list, flags
    __host__ __device__ size_t bytes() const { return doubles() * 8 + size_t(places) * (4 + 2 + 2 + 1) + 16; }
};

template <int CTRL>
__device__ __forceinline__ double quad_bcast(double v) {
    union {
        double d;
        int w[2];
    } a, r;
    a.d = v;
    r.w[0] = __builtin_amdgcn_mov_dpp(a.w[0], CTRL, 0xF, 0xF, true);
    r.w[1] = __builtin_amdgcn_mov_dpp(a.w[1], CTRL, 0xF, 0xF, true);
    return r.d;
}
// Component c (0..2) of the vector that lane LANE of this lane's quad holds.
template <int LANE>
__device__ __forceinline__ double quad_comp(d3 v, uint32_t c) {
    const double x = quad_bcast<LANE * 0x55>(v.x), y = quad_bcast<LANE * 0x55>(v.y), z = quad_bcast<LANE * 0x55>(v.z);
    return c == 0 ? x : (c == 1 ? y : z);
}

// TINY_BROKEN: a bond that broke in this step's pass, an unbonded pair from the
// next one on.
enum : uint8_t { TINY_NONE = 0, TINY_FREE, TINY_CONTACT, TINY_BOND, TINY_BROKEN, TINY_LEGACY };

template <int BIN, int HAM>
__global__ void __launch_bounds__(kTinyThreads)
    k_tiny_steps(hg_params P, sys_view S, double *gx, double *gv, double *gth, double *gw, facet_dev *facets,
                 uint32_t nsteps, double half, double dt, int nf_advance, double *lconn, uint32_t maxb) {
    extern __shared__ double tiny_lds[];
    __shared__ facet_dev F[kMaxFacets];
    __shared__ uint32_t s_bonds, s_touch;
    __shared__ uint32_t s_spare;  // with no more touching pairs than this no row overflows
    __shared__ uint32_t s_cnt[kTinySystemMax], s_legacy[kTinySystemMax];  // partners and legacy bonds
    __shared__ uint32_t s_carried[kTinySystemMax];  // row entries of partners that are not listed
    const tiny_layout Y(S.n, maxb);
    const uint32_t n = Y.n, row = Y.row, places = Y.places, tid = threadIdx.x;
    const bool nl = P.pair_mode == HG_PAIRS_NEIGHBOR_LIST;
    double *X = tiny_lds;                        // 18 components of n
    double *T = X + size_t(18) * n;              // 6 components of every place
    double *SP = T + size_t(6) * places;         // 9 components of every place
    double *FT = SP + size_t(9) * places;        // 6 components of n
    double *C = FT + size_t(6) * n;              // connectors: 15 per (particle, bond slot)
    uint32_t *E = reinterpret_cast<uint32_t *>(C + size_t(15) * maxb * n);  // i | j << 8 | legacy slots: i's << 16, j's << 24
    uint16_t *LB = reinterpret_cast<uint16_t *>(E + places), *LC = LB + places;
    uint8_t *K = reinterpret_cast<uint8_t *>(LC + places);
    auto vec = [&](uint32_t f, uint32_t i) {
        const double *q = X + size_t(3 * f) * n + i;
        return d3{q[0], q[n], q[2 * n]};
    };
    auto spring = [&](uint32_t at, uint32_t c) {
        const double *q = SP + size_t(3 * c) * places + at;
        return d3{q[0], q[places], q[2 * places]};
    };
    auto set_spring = [&](uint32_t at, uint32_t c, d3 a) {
        double *q = SP + size_t(3 * c) * places + at;
        q[0] = a.x;
        q[places] = a.y;
        q[2 * places] = a.z;
    };

    // in: state, facets, connectors, then the pairs with their springs
    const double *fields[6] = {gx, gv, gw, gth, S.a, S.al};
    for (uint32_t q = tid; q < 18u * n; q += kTinyThreads) {
        const uint32_t c = q / n, i = q % n;
        X[q] = fields[c / 3][4 * i + c % 3];
    }
    if (tid < uint32_t(S.nf)) F[tid] = facets[tid];
    if (tid == 0) {
        s_bonds = s_touch = 0;
        s_spare = S.pt.cap + 1 < n ? S.pt.cap : kNoEntry;
    }
    if (tid < n) {
        s_cnt[tid] = nl ? S.ncnt[tid] : n - 1u;
        s_legacy[tid] = BIN == HG_BINARY_SINTER_LEGACY ? S.pt.bcnt[tid] : 0u;
        s_carried[tid] = BIN != HG_BINARY_NONE ? S.pt.pcnt_old[tid] : 0u;
    }
    if constexpr (BIN == HG_BINARY_SINTER_LEGACY)
        for (uint32_t q = tid; q < 15u * maxb * n; q += kTinyThreads) {
            const uint32_t e = q / 15, i = e / maxb, s = e % maxb;
            C[q] = lconn[(size_t(s) * n + i) * kConnRec + q % 15];
        }
    __syncthreads();
    for (uint32_t at = tid; at < places; at += kTinyThreads) {
        const uint32_t i = at / row, k = at % row;
        const bool on = k < s_cnt[i];
        uint8_t kind = TINY_NONE;
        if (on) {
            const uint32_t j = nl ? S.nb[size_t(k) * n + i] : k + (k >= i ? 1u : 0u);
            uint32_t ls = 0;
            kind = TINY_FREE;
            if constexpr (BIN == HG_BINARY_SINTER_LEGACY)
                for (uint32_t q = 0; q < s_legacy[i]; q++)
                    if (S.pt.bj[size_t(q) * n + i] == j) {
                        kind = TINY_LEGACY;
                        ls = q | (S.pt.lslot[size_t(q) * n + i] << 8);
                    }
            E[at] = i | (j << 8) | (ls << 16);
            if constexpr (BIN != HG_BINARY_NONE) {
                const uint32_t cnt = S.pt.pcnt_old[i];
                for (uint32_t q = 0; q < cnt; q++) {
                    const uint32_t tag = S.pt.pj_old[size_t(q) * n + i];
                    if ((tag & kIdxMask) != j) continue;
                    kind = (tag & kBondBit) ? TINY_BOND : TINY_CONTACT;
                    atomicSub(&s_carried[i], 1u);
                    const spring9 sp = ld_rec(S.pt.ps_old + (size_t(q) * n + i) * kSpringRec);
                    for (uint32_t c = 0; c < 3; c++) set_spring(at, c, sp.s[c]);
                }
            }
            if (kind == TINY_BOND || kind == TINY_LEGACY) LB[atomicAdd(&s_bonds, 1u)] = uint16_t(at);
        }
        K[at] = kind;
    }
    if (BIN != HG_BINARY_NONE && tid < n && S.pt.cap + 1 < n)
        atomicMin(&s_spare, S.pt.cap - (S.pt.pcnt_old[tid] < S.pt.cap ? S.pt.pcnt_old[tid] : S.pt.cap));
    // the first kick and drift
    for (uint32_t q = tid; q < 6u * n; q += kTinyThreads) {
        const uint32_t c = q / n, i = q % n, ang = c >= 3, d = c % 3;
        double *u = X + size_t(3 + c) * n + i, *o = X + size_t((ang ? 9 : 0) + d) * n + i;
        *u = *u + X[size_t(12 + c) * n + i] * half;
        *o = *o + *u * dt;
    }
    const contact_reach reach(P.contact.r_part);
    for (uint32_t s = 0; s < nsteps; s++) {
        __syncthreads();
        if constexpr (BIN == HG_BINARY_SINTER_LEGACY) {
            // sinter_step_handler: a connector follows its particle, then turns with it
            for (uint32_t q = tid; q < 5u * maxb * n; q += kTinyThreads) {
                const uint32_t e = q / 5, i = e / maxb;
                if (e % maxb >= s_legacy[i]) continue;
                double *r = C + size_t(3) * q;
                const d3 p = d3{r[0], r[1], r[2]} + vec(1, i) * dt;
                const d3 moved = p + cross(vec(2, i) * dt, p - vec(0, i));
                r[0] = moved.x;
                r[1] = moved.y;
                r[2] = moved.z;
            }
        }
        if constexpr (BIN != HG_BINARY_NONE)
            for (uint32_t at = tid; at < places; at += kTinyThreads) {
                const uint8_t kind = K[at];
                if (kind != TINY_FREE && kind != TINY_CONTACT && kind != TINY_BROKEN) continue;
                const uint32_t e = E[at];
                const d3 d = vec(0, e & 0xFFu) - vec(0, (e >> 8) & 0xFFu);
                bool touching = false;
                if (!reach.beyond(dot(d, d))) touching = !(2.0 * P.contact.r_part - dot(d, normalized(d)) <= 0);
                if (touching) {
                    LC[atomicAdd(&s_touch, 1u)] = uint16_t(at);
                    if (kind != TINY_CONTACT) {
                        for (uint32_t c = 0; c < 3; c++) set_spring(at, c, zero3());
                        K[at] = TINY_CONTACT;
                    }
                } else {
                    K[at] = TINY_FREE;
                }
            }
        __syncthreads();
        // terms: bonded quads, touching quads, the other pairs, facets, each
        // kind from a wavefront of its own
        const uint32_t bonds = s_bonds, touching = s_touch, spare = s_spare, per = BIN == HG_BINARY_SINTER_LEGACY ? 1u : 4u;
        const uint32_t e1 = (bonds * per + 63u) & ~63u, e2 = e1 + ((touching * 4u + 63u) & ~63u),
                       e3 = e2 + ((places + 63u) & ~63u), e4 = e3 + (S.nf > 0 ? n : 0u);
        for (uint32_t q = tid; q < e4; q += kTinyThreads) {
            if (q >= e3) {
                const uint32_t i = q - e3;
                const acc6 f = facet_fold(P, F, S.nf, S.ss, n, i, vec(0, i), vec(1, i), vec(2, i));
                const double r[6] = {f.lin.x, f.lin.y, f.lin.z, f.ang.x, f.ang.y, f.ang.z};
                for (uint32_t c = 0; c < 6; c++) FT[size_t(c) * n + i] = r[c];
            } else if (q >= e2) {
                const uint32_t at = q - e2;
                if (at >= places || K[at] != TINY_FREE) continue;
                const uint32_t e = E[at];
                const d3 h = hamaker_lin<HAM>(P.hamaker, vec(0, (e >> 8) & 0xFFu) - vec(0, e & 0xFFu));
                T[at] = h.x;
                T[places + at] = h.y;
                T[2 * places + at] = h.z;
                for (uint32_t c = 3; c < 6; c++) T[c * places + at] = 0.0;
            } else if (BIN == HG_BINARY_SINTER_LEGACY && q < e1) {
                if (q >= bonds) continue;
                const uint32_t at = LB[q], e = E[at], i = e & 0xFFu, j = (e >> 8) & 0xFFu, ls = (e >> 16) & 0xFFu;
                // sinter_bridge.h:222-223: the bond's connectors, i's at its
                // slot for j, j's at its slot for i
                const double *ri = C + (size_t(i) * maxb + ls) * 15;
                const double *rj = C + (size_t(j) * maxb + (e >> 24)) * 15;
                d3 ci[5], cj[5];
                for (int c = 0; c < 5; c++) {
                    ci[c] = d3{ri[3 * c], ri[3 * c + 1], ri[3 * c + 2]};
                    cj[c] = d3{rj[3 * c], rj[3 * c + 1], rj[3 * c + 2]};
                }
                const acc6 b = legacy_bonded_eval(P.sinter.k, P.sinter.gamma_n, P.contact.r_part, P.contact.mass,
                                                  P.contact.inertia, ci, cj, vec(0, i), vec(0, j), vec(1, i), vec(1, j),
                                                  vec(2, i), vec(2, j));
                d3 lin = b.lin;
                if constexpr (HAM != HG_HAMAKER_NONE) lin = lin + hamaker_lin<HAM>(P.hamaker, vec(0, j) - vec(0, i));
                const double r[6] = {lin.x, lin.y, lin.z, b.ang.x, b.ang.y, b.ang.z};
                for (uint32_t c = 0; c < 6; c++) T[c * places + at] = r[c];
            } else if constexpr (BIN == HG_BINARY_CONTACT || BIN == HG_BINARY_SINTER || BIN == HG_BINARY_SINTER_LEGACY) {
                const bool bond = BIN == HG_BINARY_SINTER && q < e1;
                const uint32_t item = (bond ? q : q - e1) >> 2, c = q & 3u;
                if (item >= (bond ? bonds : touching)) continue;
                const uint32_t at = bond ? LB[item] : LC[item], e = E[at], i = e & 0xFFu, j = (e >> 8) & 0xFFu;
                if (bond && K[at] != TINY_BOND) continue;  // broken: the pair is among the others
                const d3 xi = vec(0, i), xj = vec(0, j), vi = vec(1, i), vj = vec(1, j), wi = vec(2, i), wj = vec(2, j);
                const hg_contact_params &pc = P.contact;
                const hg_sinter_params &ps = P.sinter;
                const double r = bond ? ps.r_part : pc.r_part;
                const d3 d = xi - xj, nn = normalized(d);
                const double overlap = 2.0 * r - dot(d, nn), rpp = r - overlap / 2.0, v_n = -dot(vi - vj, nn);
                const double f_n = (bond ? ps.k : pc.k) * overlap + (bond ? ps.gamma_n : pc.gamma_n) * v_n;
                const d3 cwi = cross(nn, wi), cwj = cross(nn, wj);
                const d3 v_ij = ((vi - vj) + rpp * cwi) + rpp * cwj;
                const d3 v_t = v_ij - dot(v_ij, nn) * nn, v_r = (-rpp) * (cwi - cwj),
                         v_o = (r * (dot(nn, wi) - dot(nn, wj))) * nn;
                auto pick = [&](auto a, auto b, auto o) { return c == 0 ? a : (c == 1 ? b : o); };
                const d3 rel{pick(v_t.x, v_r.x, v_o.x), pick(v_t.y, v_r.y, v_o.y), pick(v_t.z, v_r.z, v_o.z)};
                d3 f;
                if (c == 3) {
                    f = hamaker_lin<HAM>(P.hamaker, xj - xi);
                } else {
                    d3 sp = spring(at, c);
                    if (bond)
                        f = shear_sinter(sp, nn, pick(ps.k_t, ps.k_r, ps.k_o), pick(ps.gamma_t, ps.gamma_r, ps.gamma_o),
                                         rel, ps.dt);
                    else
                        f = shear_contact(sp, nn, pick(pc.k_t, pc.k_r, pc.k_o), pick(pc.gamma_t, pc.gamma_r, pc.gamma_o),
                                          f_n, pick(pc.mu_s, pc.mu_r, pc.mu_o), pick(pc.phi_d, pc.phi_r, pc.phi_o), rel,
                                          pc.dt);
                    set_spring(at, c, sp);
                }
                const d3 cr = cross(nn, f);
                const d3 tau = c == 0 ? rpp * cr : (c == 1 ? r * cr : r * f);
                const double ft = quad_comp<0>(f, c), h = quad_comp<3>(f, c), tt = quad_comp<0>(tau, c),
                             tr = quad_comp<1>(tau, c), to = quad_comp<2>(tau, c);
                if (bond && P.sinter_breaking) {
                    // alt_breaking_sinter_bridge.h:117-119; lane 0 holds f_t
                    const d3 ftot = f_n * nn + f;
                    if (c == 0) {
                        double neck = __builtin_huge_val();
                        if (S.pt.bcnt)
                            for (uint32_t b = 0; b < S.pt.bcnt[i]; b++)
                                if (S.pt.bj[size_t(b) * n + i] == j) neck = S.pt.bstr[size_t(b) * n + i];
                        if (norm(ftot) > neck) K[at] = TINY_BROKEN;
                    }
                }
                if (c < 3) {
                    const double nc = c == 0 ? nn.x : (c == 1 ? nn.y : nn.z);
                    double lin = (f_n * nc + ft) / (bond ? ps.mass : pc.mass);
                    if constexpr (HAM != HG_HAMAKER_NONE) lin = lin + h;
                    T[c * places + at] = lin;
                    T[(3 + c) * places + at] = ((-tt + tr) + to) / (bond ? ps.inertia : pc.inertia);
                }
            }
        }
        __syncthreads();
        if (tid == 0) {
            s_touch = 0;
            advance_facets(F, nf_advance, dt);
        }
        // a row that holds more entries than the table, if only for this step, is
        // reported as the walk reports it; threads that the sums leave idle
        const uint32_t ri = tid - kTinyThreads / 2;
        if (BIN != HG_BINARY_NONE && __builtin_expect(touching > spare, 0) && ri < n) {
            uint32_t held = s_carried[ri];
            for (uint32_t k = 0; k < s_cnt[ri]; k++) {
                const uint8_t kind = K[ri * row + k];
                held += kind == TINY_CONTACT || kind == TINY_BOND ? 1u : 0u;
            }
            if (held > S.pt.cap) {
                atomicOr(&S.flags[FLAG_PAIR_OVERFLOW], 1);
                atomicMax(&S.flags[FLAG_PAIR_MAXCOUNT], int(held));
            }
        }
        // sums in partner order, then the kicks and the drift, a component a thread
        const bool last = s + 1 == nsteps;
        for (uint32_t q = tid; q < 6u * n; q += kTinyThreads) {
            const uint32_t c = q / n, i = q % n, ang = c >= 3, d = c % 3;
            const uint32_t m = s_cnt[i];
            const double *t = T + size_t(c) * places + size_t(i) * row;
            double acc = 0.0;
#pragma unroll 6
            for (uint32_t k = 0; k < m; k++) acc = acc + t[k];
            if (S.nf > 0) acc = acc + FT[q];
            double *u = X + size_t(3 + c) * n + i, *o = X + size_t((ang ? 9 : 0) + d) * n + i;
            double w = *u + acc * half;
            if (last) {
                X[size_t(12 + c) * n + i] = acc;
            } else {
                w = w + acc * half;
                *o = *o + w * dt;
            }
            *u = w;
        }
    }
    __syncthreads();
    double *back[6] = {gx, gv, gw, gth, S.a, S.al};
    for (uint32_t q = tid; q < 18u * n; q += kTinyThreads) {
        const uint32_t c = q / n, i = q % n;
        back[c / 3][4 * i + c % 3] = X[q];
        if (c >= 3 && c < 9 && !__builtin_isfinite(X[q])) atomicOr(&S.flags[FLAG_NUMERIC], 1);
    }
    if (tid < uint32_t(S.nf)) facets[tid] = F[tid];
    if constexpr (BIN == HG_BINARY_SINTER_LEGACY)
        for (uint32_t q = tid; q < 15u * maxb * n; q += kTinyThreads) {
            const uint32_t e = q / 15, i = e / maxb, s = e % maxb;
            if (s < S.pt.bcnt[i]) lconn[(size_t(s) * n + i) * kConnRec + q % 15] = C[q];
        }
    // the rows as the walk leaves them: entries of partners not listed carried in place
    if constexpr (BIN != HG_BINARY_NONE) {
        if (tid < n) {
            const uint32_t i = tid, cnt_old = S.pt.pcnt_old[i], m = s_cnt[i];
            uint32_t q = 0, p = 0;
            auto put = [&](uint32_t tag, const spring9 &sp) {
                if (q < S.pt.cap) {
                    S.pt.pj_new[size_t(q) * n + i] = tag;
                    st_rec(S.pt.ps_new + (size_t(q) * n + i) * kSpringRec, sp);
                }
                q++;
            };
            auto carry_below = [&](uint32_t j) {
                while (p < cnt_old && (S.pt.pj_old[size_t(p) * n + i] & kIdxMask) < j) {
                    put(S.pt.pj_old[size_t(p) * n + i], ld_rec(S.pt.ps_old + (size_t(p) * n + i) * kSpringRec));
                    p++;
                }
            };
            for (uint32_t k = 0; k < m; k++) {
                const uint32_t at = i * row + k, j = (E[at] >> 8) & 0xFFu;
                carry_below(j);
                if (p < cnt_old && (S.pt.pj_old[size_t(p) * n + i] & kIdxMask) == j) p++;  // replaced
                if (K[at] == TINY_CONTACT || K[at] == TINY_BOND)
                    put(j | (K[at] == TINY_BOND ? kBondBit : 0u),
                        spring9{{spring(at, 0), spring(at, 1), spring(at, 2)}});
            }
            carry_below(kNoEntry & kIdxMask);
            S.pt.pcnt_new[i] = q < S.pt.cap ? q : S.pt.cap;
            if (q > S.pt.cap) {
                atomicOr(&S.flags[FLAG_PAIR_OVERFLOW], 1);
                atomicMax(&S.flags[FLAG_PAIR_MAXCOUNT], int(q));
            }
        }
    }
}

bool tiny_steps_fit(uint32_t n, uint32_t maxb) { return tiny_layout(n, maxb).bytes() <= size_t(154) * 1024; }

template <int BIN, int HAM>
hipError_t launch_small_steps_t(const hg_params &p, const sys_view &even, const sys_view &odd, double *x, double *v,
                                double *th, double *w, facet_dev *facets, uint32_t nsteps, double half, double dt,
                                int nf_advance, double *lconn, const uint32_t *bcnt, uint32_t maxb, hipStream_t s) {
    if (even.n <= kTinySystemMax && tiny_steps_fit(even.n, maxb)) {
        const uint32_t bytes = uint32_t(tiny_layout(even.n, maxb).bytes());
        const auto kernel = &k_tiny_steps<BIN, HAM>;
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
        if (e != hipSuccess) return e;
        kernel<<<1, kTinyThreads, bytes, s>>>(p, even, x, v, th, w, facets, nsteps, half, dt, nf_advance, lconn, maxb);
        return hipGetLastError();
    }
    if constexpr (BIN == HG_BINARY_SINTER_LEGACY) {
        k_small_steps<BIN, HAM><<<1, kTile, 0, s>>>(p, even, odd, x, v, th, w, facets, nsteps, half, dt, nf_advance,
                                                    lconn, bcnt);
        return hipGetLastError();
    }
    return hipErrorInvalidValue;
}

hipError_t launch_small_steps(const hg_params &p, const sys_view &even, const sys_view &odd, double *x, double *v,
                              double *th, double *w, facet_dev *facets, uint32_t nsteps, double half, double dt,
                              int nf_advance, double *lconn, const uint32_t *bcnt, uint32_t maxb, hipStream_t s) {
    if (even.n == 0 || even.n > kSmallSystemMax || p.precision != HG_PRECISION_FP64) return hipErrorInvalidValue;
#define HG_CASE(B, H)                                                                                                \
    if (p.binary_model == B && p.hamaker_model == H)                                                                 \
        return launch_small_steps_t<B, H>(p, even, odd, x, v, th, w, facets, nsteps, half, dt, nf_advance, lconn, bcnt, \
                                          maxb, s);
    HG_CASE(HG_BINARY_NONE, HG_HAMAKER_NONE)
    HG_CASE(HG_BINARY_NONE, HG_HAMAKER_FULL)
    HG_CASE(HG_BINARY_NONE, HG_HAMAKER_LIMITED)
    HG_CASE(HG_BINARY_NONE, HG_HAMAKER_SIMPLIFIED)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_NONE)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_FULL)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_LIMITED)
    HG_CASE(HG_BINARY_CONTACT, HG_HAMAKER_SIMPLIFIED)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_NONE)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_FULL)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_LIMITED)
    HG_CASE(HG_BINARY_SINTER, HG_HAMAKER_SIMPLIFIED)
    HG_CASE(HG_BINARY_SINTER_LEGACY, HG_HAMAKER_NONE)
    HG_CASE(HG_BINARY_SINTER_LEGACY, HG_HAMAKER_FULL)
    HG_CASE(HG_BINARY_SINTER_LEGACY, HG_HAMAKER_LIMITED)
    HG_CASE(HG_BINARY_SINTER_LEGACY, HG_HAMAKER_SIMPLIFIED)
#undef HG_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_kick_drift(double *x, double *v, double *th, double *w, const double *a, const double *al,
                             uint32_t n, bool pending, double half_prev, double half, double dt, facet_dev *facets,
                             int nf, double facet_dt, hipStream_t s) {
    unsigned nb = blocks_for(n > 0 ? n : 1, 256);
    k_kick_drift<<<nb, 256, 0, s>>>(x, v, th, w, a, al, n, pending ? 1 : 0, half_prev, half, dt, facets, nf,
                                    facet_dt);
    return hipGetLastError();
}

hipError_t launch_legacy_move(const double *x, const double *v, const double *w, uint32_t n, double dt,
                              double *lconn, const uint32_t *bcnt, hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_legacy_move<<<blocks_for(n, 256), 256, 0, s>>>(x, v, w, n, dt, lconn, bcnt);
    return hipGetLastError();
}

hipError_t launch_final_kick(double *v, double *w, const double *a, const double *al, uint32_t n, double half,
                             facet_dev *facets, int nf, double facet_dt, int *flags, hipStream_t s) {
    unsigned nb = blocks_for(n > 0 ? n : 1, 256);
    k_final_kick<<<nb, 256, 0, s>>>(v, w, a, al, n, half, facets, nf, facet_dt, flags);
    return hipGetLastError();
}

hipError_t launch_advance_facet(facet_dev *f, const double *v, double dt, hipStream_t s) {
    k_advance_facet<<<1, 64, 0, s>>>(f, v[0], v[1], v[2], dt);
    return hipGetLastError();
}

hipError_t launch_zero_u32(uint32_t *p, size_t count, hipStream_t s) {
    if (count == 0) return hipSuccess;
    unsigned nb = unsigned(std::min<size_t>(1024, (count + 255) / 256));
    k_zero_u32<<<nb, 256, 0, s>>>(p, count);
    return hipGetLastError();
}

hipError_t launch_copy_words(const int *src, int *dst, int count, hipStream_t s) {
    k_copy_words<<<1, 64, 0, s>>>(src, dst, count);
    return hipGetLastError();
}

hipError_t launch_pack3(const double *const *src, int count, size_t n, double *out, hipStream_t s) {
    if (count == 0 || n == 0) return hipSuccess;
    pack_src F{};
    for (int k = 0; k < count; k++) F.f[k] = src[k];
    const unsigned nb = unsigned(std::min<size_t>(512, (3 * n + 255) / 256));
    k_pack3<<<dim3(nb, unsigned(count)), 256, 0, s>>>(F, 3 * n, out);
    return hipGetLastError();
}

hipError_t launch_zero_f64(double *p, size_t count, hipStream_t s) {
    if (count == 0) return hipSuccess;
    unsigned nb = unsigned(std::min<size_t>(1024, (count + 255) / 256));
    k_zero_f64<<<nb, 256, 0, s>>>(p, count);
    return hipGetLastError();
}

hipError_t launch_exclusive_scan(const uint32_t *in, uint32_t *out, uint32_t count, uint32_t *tmp, hipStream_t s) {
    if (count == 0) return hipSuccess;
    const uint32_t nblocks = (count + kScanChunk - 1) / kScanChunk;
    k_scan_blocks<<<nblocks, kScanThreads, 0, s>>>(in, out, count, tmp);
    k_scan_top<<<1, kScanThreads, 0, s>>>(tmp, nblocks);
    k_scan_add<<<nblocks, kScanThreads, 0, s>>>(out, count, tmp);
    return hipGetLastError();
}

uint32_t scan_tmp_words(uint32_t count) { return (count + kScanChunk - 1) / kScanChunk + 1; }

hipError_t launch_cell_lists(const list_build &B, hipStream_t s) {
    if (B.count == 0) return hipSuccess;
    const double cs = 2.0 * B.r_verlet * (1.0 + 1e-9);  // two list radii: 2 x 2 x 2 cells per particle
    hipError_t e;
    if ((e = launch_zero_u32(B.buckets, size_t(2) * B.hash_size, s)) != hipSuccess) return e;
    k_cell_count<<<blocks_for(B.count, 256), 256, 0, s>>>(B, cs);
    if ((e = launch_exclusive_scan(B.buckets, B.bucket_start, B.hash_size, B.scan_tmp, s)) != hipSuccess) return e;
    k_cell_fill<<<blocks_for(B.count, 256), 256, 0, s>>>(B);
    k_list_fill<<<blocks_for(B.count, kListParts), 256, 0, s>>>(B, cs);
    return hipGetLastError();
}

hipError_t launch_neighbor_build(hg_system_impl &S, hipStream_t s) {
    const uint32_t n = uint32_t(S.n);
    if (n == 0) return hipSuccess;
    const list_build B{S.x,       n,            S.n,        S.p.r_verlet, nullptr,     nullptr,
                       S.hash_size, S.buckets, S.bucket_start, S.scan_tmp, S.cell_of,  S.cell_recs, S.nb,
                       S.ncnt,      S.cap_n,   S.flags,        nullptr};
    if (n > kBruteListMax) return launch_cell_lists(B, s);
    k_list_brute<<<blocks_for(n, kBruteParts), 256, 0, s>>>(B);
    return hipGetLastError();
}

hipError_t launch_diagnostics(const double *x, const double *v, const double *w, uint32_t n, double mass,
                              double inertia, double *out, hipStream_t s) {
    k_diag<<<1, 1024, 0, s>>>(x, v, w, n, mass, inertia, out);
    return hipGetLastError();
}

hipError_t launch_energy(const hg_params &p, const energy_view &E, double mass, double inertia, double *out,
                         hipStream_t s) {
    if (E.n == 0) return hipSuccess;
    k_energy<<<blocks_for(8 * size_t(E.n), 256), 256, 0, s>>>(p, E, mass, inertia, out);
    return hipGetLastError();
}

}  // namespace hg

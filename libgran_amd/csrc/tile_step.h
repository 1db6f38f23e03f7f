// Per-step kernels over many workgroups: one launch per time step for a whole
// set of systems (the wide systems of a pool, or one hg_system), each
// workgroup carrying a tile of W particles.
//
// One lane per particle walking its partners in turn leaves most of the chip
// idle at the sizes a single aggregate has (20,000 particles are 313
// wavefronts for 1,024 SIMDs) and makes a step as long as the longest chain of
// dependent pair evaluations. Here a workgroup spreads its tile's ordered
// pairs over all its threads: the listed partners are read k by k, matched
// against the particle's table row and queued in LDS, bonded pairs apart from
// the others, so that a wavefront evaluates one kind; each pair leaves its
// term in LDS at its place in the list, and one thread per particle adds the
// terms in list order, which gives the sums of the walk bit for bit. The same
// thread then completes the step and drifts the particle into the other set
// of x, v, omega buffers (other workgroups still read this one), so a step is
// one launch.
//
// The pair-state rows are updated in place: a spring goes back to the slot it
// came from. A row changes only when a contact begins or ends (or a bond
// breaks). Its owner thread fills the slot of an ended entry with the row's last
// one, and new entries go to the row's end; in the last launch of an interval it
// puts a row that is out of order in order, so the table is canonical whenever
// anything but these launches reads it. Kept in order in every launch, a bed's
// rows of twelve moved several records for each contact that began or ended: a
// face-centred packing of 32,000, mixed, lists of 12, took 47 us a step, 32 so
// (the walk of one lane a particle 42). A row that is full when a contact begins may lose an entry to a
// later part of the list: the new entry waits in the table's other half, which
// these launches leave alone, and a row overflows only if it still waits at the
// end.
#pragma once

#include "pair_eval.h"
#include "pool_device.h"

namespace hg {

namespace {

// LDS of a tile: own state, the terms of KC list positions per particle
// (position kk of particle i at [kk * W + i]), the queue of those positions'
// pairs, and the rows' counts.
template <int W, int KC, int PREC, bool FAC>
struct tile_lds {
    using term = typename prec_types<PREC>::term;
    static_assert(KC * W <= int(kTilePlaces), "queue_word");
    double s[12][W];  // x, v, omega, theta
    term T[6][KC * W];
    uint2 Q[KC * W];  // partner and queue_word
    uint16_t CW[KC * W];
    uint32_t rows[W], dirty[W];  // lengths; whether entries ended or began in this part of the lists
    // slots of ended entries (kManyHoles: others from slot 31 on); the length
    // without them of a row that has some
    uint32_t holes[W], kept[W];
    uint32_t more[W], spilled;  // a row's entries in the table's other half, and whether there are any
    uint32_t nB[kTileThreads / 64], nO[kTileThreads / 64];
    uint32_t contacts, ended;
    // the terms of four facets: FP64 the 6 components of each, mixed the
    // contact's 6 and the Hamaker term's 3
    term F[FAC ? 4 : 1][FAC ? 9 : 1][FAC ? W : 1];
    term A[6][W < 64 ? W : 1];
};

constexpr uint32_t kManyHoles = 1u << 31;

// This workgroup's tile: from the map or, without one, of the view's only
// system, so that a single system's tile waits for no load.
__device__ __forceinline__ wide_block tile_block(const wide_block *map, const pool_view &V, uint32_t width) {
    return map ? map[blockIdx.x] : wide_block{0, blockIdx.x * width, 0, V.alone};
}

// Wavefronts per SIMD that the registers leave room for. Listed tiles, many to
// a CU, hide one pair's latency behind another's: mixed 151 us a step at
// 635,000 particles with three, 187 with two (four spill: 241); with the facet
// terms three spill too: 24 plate tests of 1,000 steps 40.5 ms, 35.8 with two.
// In FP64 nine registers spill with three, which pays where a CU has a third
// workgroup to put beside two (kTwoOnEachCu). All pairs in FP64 or with facets
// are not held to any: two, asked for, cost 33 us a step at 522 particles against
// 28. Mixed ones without facets fit three with a few registers to spare or
// spilled, and take 10.1 ms a step at 24,000 particles with two, 7.2 with three.
constexpr int tile_waves(int pairs, int prec, bool fac) {
    if (prec == HG_PRECISION_MIXED && !fac) return 3;
    return pairs != HG_PAIRS_NEIGHBOR_LIST ? 1 : 2;
}

// FP64 tiles with a binary functor and no facets in more workgroups than this are
// held to three wavefronts per SIMD: what 256 CUs take two each of. Aggregates
// with lists of 3.9 at 450 tiles 13.6 us a step with two, 14.3 with three; 550
// 17.2 and 15.2; 1,000 22.4 and 22.3; 2,500 47.4 and 42.4. Beds with lists of
// about 50 at 450 114 and 118, 600 175 and 141, 4,700 951 and 792, where the walk
// takes 824. Without a binary functor the two take the same time.
constexpr unsigned kTwoOnEachCu = 512;

// A launch's arguments (the parameter set, its mixed form and two views, 1.5 KB)
// lie in memory that no cache holds yet. Read where they are used, they were
// three or four round trips one after the other, 4,400 cycles; one word of each
// 64-byte line read together at the start brings them all in for 1,250.
template <size_t BYTES>
__device__ __forceinline__ void touch_args() {
    using words = const __attribute__((address_space(4))) uint32_t;
    words *a = (words *)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t any = 0;
#pragma unroll
    for (size_t q = 0; q < BYTES / 4; q += 16) any |= a[q];
    asm volatile("" ::"s"(any));
}

// What a launch does after the pass: TILE_FORCE stores the accelerations of
// the systems that have none; TILE_STEP completes the step, kicks and drifts
// into the other buffers; TILE_LAST completes the last step.
template <int BIN, int HAM, int PAIRS, int PREC, bool FAC, int PER_SIMD = tile_waves(PAIRS, PREC, FAC)>
__global__ void __launch_bounds__(kTileThreads, PER_SIMD)
    k_tile_step(hg_params P, mixed_consts MC, pool_view Vi, pool_view Vo, const wide_block *map, int mode, double half,
                double dt) {
    constexpr int W = tile_width(PAIRS), KC = tile_depth(PAIRS), ROWS = kTileThreads / W, WAVES = kTileThreads / 64;
    using term = typename prec_types<PREC>::term;
    using vec = typename prec_types<PREC>::vec;
    __shared__ tile_lds<W, KC, PREC, FAC> L;
    // a workgroup is a wavefront for each SIMD: the CU's LDS holds as many
    static_assert(sizeof(L) * size_t(PER_SIMD) <= 160u * 1024u, "LDS of the tiles on a CU");
    touch_args<sizeof(hg_params) + sizeof(mixed_consts) + 2 * sizeof(pool_view)>();
    const wide_block b = tile_block(map, Vi, W);
    const uint32_t n = b.n & kIdxMask, cur = b.n >> 31, base = b.offset + b.start;
    const uint32_t nt = n - b.start < uint32_t(W) ? n - b.start : uint32_t(W);
    const uint32_t tid = threadIdx.x, wv = tid >> 6, lane = tid & 63u;
    if (mode == TILE_FORCE && Vi.meta[b.slot].acc_valid) return;
    const size_t stride = Vi.stride;
    uint32_t *pj = cur ? Vi.pj1 : Vi.pj0, *pcnt = cur ? Vi.pcnt1 : Vi.pcnt0;
    double *ps = cur ? Vi.ps1 : Vi.ps0;
    const pair_eval<HAM, PREC> ev(P, MC);

    const uint32_t i = tid % W, r0 = tid / W;  // own particle of the tile, first list row
    const uint32_t g = base + (i < nt ? i : 0);
    // Everything that only the tile's place tells is loaded in one go: counts,
    // tags, the first part of the list (whatever its length) and the state. With
    // tags and list loaded once the counts and the state were there, they took
    // another round trip or two of some 1,700 cycles. With the arguments above,
    // the list's depth of 12 and the sums below: 200 particles, 500 steps 4.42 ->
    // 3.98 ms; 213,000 in 333 systems, FP64, 76.6 -> 71.5 ms.
    uint32_t cnt = n - 1u, c_old = 0;
    if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) cnt = Vi.ncnt[g];
    if constexpr (BIN != HG_BINARY_NONE) c_old = pcnt[g];
    uint32_t tags[4], js[KC / ROWS];
    if constexpr (BIN != HG_BINARY_NONE) {
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) tags[s] = pj[size_t(s < Vi.cap_s ? s : 0u) * stride + g];
    }
    if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) {
#pragma unroll
        for (uint32_t q = 0; q < KC / ROWS; q++) {
            const uint32_t k = r0 + q * ROWS;
            js[q] = Vi.nb[size_t(k < Vi.cap_n ? k : 0u) * stride + g];
        }
    }
    if (r0 < 4) {
        const d3 a = ld3(r0 == 0 ? Vi.x : (r0 == 1 ? Vi.v : (r0 == 2 ? Vi.w : Vi.th)), g);
        L.s[3 * r0][i] = a.x;
        L.s[3 * r0 + 1][i] = a.y;
        L.s[3 * r0 + 2][i] = a.z;
    }
    if (i >= nt) cnt = c_old = 0;
    if (tid < uint32_t(W)) {
        L.rows[tid] = c_old;
        L.dirty[tid] = L.holes[tid] = L.more[tid] = 0;
        L.kept[tid] = kNoEntry;
    }
    if (tid == 0) L.contacts = L.ended = L.spilled = 0;
    auto own = [&](int f, uint32_t t) { return d3{L.s[3 * f][t], L.s[3 * f + 1][t], L.s[3 * f + 2][t]}; };

    // Facets f0 .. f0 + 3, one per wavefront (W == 64) or thread group: their
    // terms to LDS, where fold_facets adds them to the right fold over f.
    const uint32_t nf = FAC ? Vi.meta[b.slot].nf : 0u;
    auto facet_terms = [&](uint32_t f0) {
        if constexpr (FAC) {
            const uint32_t q = W == 64 ? wv : r0, f = f0 + q;
            if (q < 4 && f < nf && i < nt) {
                const facet_dev fd = Vi.facets[size_t(b.slot) * Vi.max_facets + f];
                auto put = [&](uint32_t c, vec u) {
                    L.F[q][c][i] = u.x;
                    L.F[q][c + 1][i] = u.y;
                    L.F[q][c + 2][i] = u.z;
                };
                if constexpr (PREC == HG_PRECISION_FP64) {
                    const acc6 e = facet_term(P, fd, int(f), Vi.ss, stride, g, own(0, i), own(1, i), own(2, i));
                    put(0, e.lin);
                    put(3, e.ang);
                } else {
                    accf c;
                    f3 h;
                    facet_term_mx(P, MC, fd, int(f), Vi.ss, stride, g, own(0, i), own(1, i), own(2, i), c, h);
                    put(0, c.lin);
                    put(3, c.ang);
                    put(6, h);
                }
            }
        }
    };
    vec fsum{};  // rows 0 and 1: this thread's half (force, torque) of the fold so far
    auto fold_facets = [&](uint32_t f0) {
        if constexpr (FAC) {
            if (r0 >= 2) return;
            for (int f = int(min(f0 + 4u, nf)) - 1; f >= int(f0); f--) {
                const auto &t = L.F[f - int(f0)];
                const vec e{t[3 * r0][i], t[3 * r0 + 1][i], t[3 * r0 + 2][i]};
                if constexpr (PREC == HG_PRECISION_FP64) {
                    fsum = f == int(nf) - 1 ? e : e + fsum;
                } else {
                    if (P.facet_contact) fsum = fsum + e;
                    if (P.facet_hamaker && r0 == 0) fsum = fsum + vec{t[6][i], t[7][i], t[8][i]};
                }
            }
        }
    };
    if constexpr (FAC) {
        if (nf > 4) {  // all but the first four ahead of the pairs
            __syncthreads();
            for (uint32_t f0 = (nf - 1) & ~3u; f0 > 0; f0 -= 4) {
                facet_terms(f0);
                __syncthreads();
                fold_facets(f0);
                __syncthreads();
            }
        }
    }

    const uint32_t seg = wv * 64u * (KC / ROWS);  // this wavefront's part of the queue
    bool unsorted = false;  // the particle's row, by this launch or those before it
    uint32_t waiting = 0;   // its owner's copy of L.more
    // an entry that ends in the evaluation
    auto end_entry = [&](uint32_t t, uint32_t slot) {
        if (slot < 31u) {
            atomicOr(&L.holes[t], 1u << slot);
        } else {
            pj[size_t(slot) * stride + base + t] = kNoEntry;
            atomicOr(&L.holes[t], kManyHoles);
        }
        L.dirty[t] = L.ended = 1;
    };
    vec accv{};          // W == 64: wavefront 0 sums forces, wavefront 1 torques
    term acct = term(0);  // W < 64: thread c * W + i sums component c
    for (uint32_t k0 = 0;; k0 += KC) {
        // queue the pairs of list positions k0 .. k0 + KC - 1: bonded ones
        // from the front of the wavefront's part, the others from its back
        if constexpr (BIN != HG_BINARY_NONE) {
#pragma unroll
            for (uint32_t s = 0; s < 4; s++)
                if (s >= c_old) tags[s] = kNoEntry;
        }
#pragma unroll
        for (uint32_t q = 0; q < KC / ROWS; q++) {
            const uint32_t k = k0 + r0 + q * ROWS;
            if constexpr (PAIRS != HG_PAIRS_NEIGHBOR_LIST) js[q] = b.offset + k + (k >= b.start + i ? 1u : 0u);
            if (k >= cnt) js[q] = kNoEntry;
        }
        // each pair's row entry: its slot, the bond bit above it
        uint32_t held[KC / ROWS];
#pragma unroll
        for (uint32_t q = 0; q < KC / ROWS; q++) held[q] = kNoRowSlot;
        if constexpr (BIN != HG_BINARY_NONE) {
            auto match = [&](const uint32_t (&t)[4], uint32_t s0) {
#pragma unroll
                for (uint32_t q = 0; q < KC / ROWS; q++)
#pragma unroll
                    for (uint32_t s = 0; s < 4; s++)
                        if ((t[s] & kIdxMask) == js[q]) held[q] = (s0 + s) | (t[s] & kBondBit);
            };
            match(tags, 0);
            uint32_t before = tags[3] & kIdxMask;
            for (uint32_t s = 1; s < 4; s++)
                unsorted |= s < c_old && (tags[s] & kIdxMask) < (tags[s - 1] & kIdxMask);
            // four at a time: one by one for every pair, with a search for every
            // contact, the bed above took 50 us
            for (uint32_t s0 = 4; s0 < c_old; s0 += 4) {
                uint32_t t[4];
#pragma unroll
                for (uint32_t s = 0; s < 4; s++) t[s] = pj[size_t(s0 + s < c_old ? s0 + s : s0) * stride + g];
#pragma unroll
                for (uint32_t s = 1; s < 4; s++)
                    if (s0 + s >= c_old) t[s] = kNoEntry;
                match(t, s0);
                for (uint32_t s = 0; s < 4 && s0 + s < c_old; s++) {
                    unsorted |= (t[s] & kIdxMask) < before;
                    before = t[s] & kIdxMask;
                }
            }
        }
        uint32_t nB = 0, nO = 0;
#pragma unroll
        for (uint32_t q = 0; q < KC / ROWS; q++) {
            const uint32_t j = js[q], slot = held[q] & kIdxMask;
            const bool on = j != kNoEntry, bond = on && (held[q] & kBondBit) != 0;
            const uint64_t mb = __ballot(on && bond), mo = __ballot(on && !bond), below = (1ull << lane) - 1ull;
            if (on) {
                const uint32_t at = bond ? nB + uint32_t(__popcll(mb & below))
                                         : 64u * (KC / ROWS) - 1u - (nO + uint32_t(__popcll(mo & below)));
                L.Q[seg + at] = uint2{j, queue_word((r0 + q * ROWS) * W + i, slot)};
            }
            nB += uint32_t(__popcll(mb));
            nO += uint32_t(__popcll(mo));
        }
        if (lane == 0) {
            L.nB[wv] = nB;
            L.nO[wv] = nO;
        }
        __syncthreads();

        // evaluate: the bonded pairs, then from the next wavefront on the others
        uint32_t tB = 0, tO = 0;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            tB += L.nB[w];
            tO += L.nO[w];
        }
        const uint32_t tBp = (tB + 63u) & ~63u;
        for (uint32_t idx = tid; idx < tBp + tO; idx += kTileThreads) {
            const bool bond = idx < tBp;
            if (bond && idx >= tB) continue;
            uint32_t rest = bond ? idx : idx - tBp, w = 0;
            for (; w + 1 < WAVES; w++) {
                const uint32_t c = bond ? L.nB[w] : L.nO[w];
                if (rest < c) break;
                rest -= c;
            }
            const uint32_t at = w * 64u * (KC / ROWS) + (bond ? rest : 64u * (KC / ROWS) - 1u - rest);
            const uint2 e = L.Q[at];
            const uint32_t pos = queue_place(e.y), t = pos % W, slot = queue_slot(e.y), j = e.x;
            const d3 xi = own(0, t), xj = ld3(Vi.x, j);
            vec lin, ang{};
            if (BIN == HG_BINARY_SINTER && bond) {
                double *rec = ps + (size_t(slot) * stride + base + t) * kSpringRec;
                spring9 sp = ld_rec(rec);
                const bool broke = ev.bonded(
                    xi, own(1, t), own(2, t), xj, ld3(Vi.v, j), ld3(Vi.w, j), sp,
                    [&] {
                        double r = __builtin_huge_val();
                        if (Vi.bcnt)
                            for (uint32_t s = 0; s < Vi.bcnt[base + t]; s++)
                                if (Vi.bj[size_t(s) * stride + base + t] == j) r = Vi.bstr[size_t(s) * stride + base + t];
                        return r;
                    },
                    lin, ang);
                st_rec(rec, sp);
                if (broke) end_entry(t, slot);
            } else {
                const bool touching = ev.template free<BIN != HG_BINARY_NONE>(xi, xj, lin);
                if constexpr (BIN != HG_BINARY_NONE) {
                    if (touching) {
                        L.CW[atomicAdd(&L.contacts, 1u)] = uint16_t(at);
                    } else if (slot != kNoRowSlot) {
                        end_entry(t, slot);
                    }
                }
            }
            L.T[0][pos] = lin.x;
            L.T[1][pos] = lin.y;
            L.T[2][pos] = lin.z;
            L.T[3][pos] = ang.x;
            L.T[4][pos] = ang.y;
            L.T[5][pos] = ang.z;
        }
        if constexpr (FAC)
            if (k0 == 0) facet_terms(0);
        __syncthreads();
        if constexpr (BIN != HG_BINARY_NONE) {
            const uint32_t nc = L.contacts;
            if (nc || L.ended) {  // uniform
                // ended entries leave their rows before new contacts claim slots,
                // the highest slot first: what is above it stays
                if (tid < nt && L.holes[tid]) {
                    const uint32_t gi = base + tid;
                    uint32_t h = L.holes[tid], c = L.rows[tid];
                    auto drop = [&](uint32_t s) {
                        if (s == --c) return;
                        pj[size_t(s) * stride + gi] = pj[size_t(c) * stride + gi];
                        st_rec(ps + (size_t(s) * stride + gi) * kSpringRec,
                               ld_rec(ps + (size_t(c) * stride + gi) * kSpringRec));
                    };
                    if (h & kManyHoles)
                        for (uint32_t s = c; s-- > 31u;)
                            if (pj[size_t(s) * stride + gi] == kNoEntry) drop(s);
                    for (h &= ~kManyHoles; h;) {
                        const uint32_t s = 31u - uint32_t(__builtin_clz(h));
                        h ^= 1u << s;
                        drop(s);
                    }
                    L.rows[tid] = L.kept[tid] = c;
                }
                __syncthreads();
                for (uint32_t c = tid; c < nc; c += kTileThreads) {
                    const uint2 e = L.Q[L.CW[c]];
                    const uint32_t pos = queue_place(e.y), t = pos % W, j = e.x, gi = base + t;
                    uint32_t slot = queue_slot(e.y);
                    const uint32_t kept = L.kept[t];
                    const d3 xj = ld3(Vi.x, j), vj = ld3(Vi.v, j), wj = ld3(Vi.w, j);
                    if (slot != kNoRowSlot && slot >= kept)  // it has moved just now
                        slot = row_slot(kept, j, [&](uint32_t s) { return pj[size_t(s) * stride + gi]; });
                    spring9 sp = zero_spring();
                    if (slot != kNoRowSlot) sp = ld_rec(ps + (size_t(slot) * stride + gi) * kSpringRec);
                    vec lin, ang;
                    ev.contact(own(0, t), own(1, t), own(2, t), xj, vj, wj, sp, lin, ang);
                    double *to = ps;
                    if (slot == kNoRowSlot) {
                        slot = atomicAdd(&L.rows[t], 1u);
                        L.dirty[t] = 1;
                        if (slot >= Vi.cap_s) {
                            slot = slot - Vi.cap_s + L.more[t];
                            L.spilled = 1;
                            if (slot < Vi.cap_s) {
                                (cur ? Vi.pj0 : Vi.pj1)[size_t(slot) * stride + gi] = j;
                                to = cur ? Vi.ps0 : Vi.ps1;
                            }
                        } else {
                            pj[size_t(slot) * stride + gi] = j;
                        }
                    }
                    if (slot < Vi.cap_s) st_rec(to + (size_t(slot) * stride + gi) * kSpringRec, sp);
                    if constexpr (HAM != HG_HAMAKER_NONE) lin = lin + vec{L.T[0][pos], L.T[1][pos], L.T[2][pos]};
                    L.T[0][pos] = lin.x;
                    L.T[1][pos] = lin.y;
                    L.T[2][pos] = lin.z;
                    L.T[3][pos] = ang.x;
                    L.T[4][pos] = ang.y;
                    L.T[5][pos] = ang.z;
                }
                __syncthreads();
                if (tid < nt && L.dirty[tid]) {
                    const uint32_t gi = base + tid;
                    uint32_t c = L.rows[tid];
                    if (L.spilled) {
                        uint32_t more = L.more[tid];
                        if (c > Vi.cap_s) {
                            more += c - Vi.cap_s;
                            c = Vi.cap_s;
                        }
                        // more than the other half holds: it overflows anyway
                        for (; c < Vi.cap_s && more > 0 && more <= Vi.cap_s; c++) {
                            more--;
                            pj[size_t(c) * stride + gi] = (cur ? Vi.pj0 : Vi.pj1)[size_t(more) * stride + gi];
                            st_rec(ps + (size_t(c) * stride + gi) * kSpringRec,
                                   ld_rec((cur ? Vi.ps0 : Vi.ps1) + (size_t(more) * stride + gi) * kSpringRec));
                        }
                        L.more[tid] = waiting = more;
                        L.rows[tid] = c;
                    }
                    pcnt[gi] = c;
                    L.dirty[tid] = L.holes[tid] = 0;
                    L.kept[tid] = kNoEntry;
                    unsorted = true;
                }
                if (tid == 0) L.contacts = L.ended = 0;
            }
        }
        // the terms of this part of the lists, in list order
        if constexpr (W == 64) {
            if (wv < 2) {
                const uint32_t left = cnt > k0 ? cnt - k0 : 0u, end = left < uint32_t(KC) ? left : uint32_t(KC);
                for (uint32_t kk = 0; kk < end; kk += 4) {  // KC is a multiple of 4
                    // a sum that starts at +0 is never -0: adding +0 for the
                    // places past a list's end changes nothing
                    vec t[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) {
                        t[u] = vec{L.T[3 * wv][(kk + u) * W + i], L.T[3 * wv + 1][(kk + u) * W + i],
                                   L.T[3 * wv + 2][(kk + u) * W + i]};
                        if (kk + u >= end) t[u] = vec{};
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4; u++) accv = accv + t[u];
                }
            }
            if (!__any(cnt > k0 + KC)) break;  // every wavefront sees the same 64 counts
        } else {
            const uint32_t all = n - 1u, left = all > k0 ? all - k0 : 0u,
                           end = left < uint32_t(KC) ? left : uint32_t(KC);
            if (tid < 6u * W) {
                // sixteen terms fetched while the sixteen before are added: the
                // adds are one chain, the fetches need not be
                term t[16], u[16];
                auto fetch = [&](term *to, uint32_t from) {
#pragma unroll
                    for (uint32_t q = 0; q < 16; q++) to[q] = L.T[r0][(from + q) * W + i];
                };
                const uint32_t full = end & ~15u;
                if (full) fetch(t, 0);
                for (uint32_t kk = 0; kk < full; kk += 16) {
                    fetch(u, kk + 16 < full ? kk + 16 : 0u);
#pragma unroll
                    for (uint32_t q = 0; q < 16; q++) {
                        acct = acct + t[q];
                        t[q] = u[q];
                    }
                }
                for (uint32_t kk = full; kk < end; kk++) acct = acct + L.T[r0][kk * W + i];
            }
            if (k0 + KC >= all) break;
        }
        __syncthreads();
        if constexpr (BIN != HG_BINARY_NONE) {
            c_old = L.rows[i];
#pragma unroll
            for (uint32_t s = 0; s < 4; s++) tags[s] = pj[size_t(s < Vi.cap_s ? s : 0u) * stride + g];
        }
        if constexpr (PAIRS == HG_PAIRS_NEIGHBOR_LIST) {
#pragma unroll
            for (uint32_t q = 0; q < KC / ROWS; q++) {
                const uint32_t k = k0 + KC + r0 + q * ROWS;
                if (k < cnt) js[q] = Vi.nb[size_t(k) * stride + g];
            }
        }
    }
    if constexpr (BIN != HG_BINARY_NONE)
        if (waiting) {
            atomicOr(&Vi.flags[FLAG_PAIR_OVERFLOW], 1);
            atomicMax(&Vi.flags[FLAG_PAIR_MAXCOUNT], int(L.rows[tid] + waiting));
            if (Vi.sflags) atomicOr(&Vi.sflags[b.slot], HG_FAULT_PAIR_CAPACITY);
        }
    if constexpr (BIN != HG_BINARY_NONE)
        if (mode != TILE_STEP && unsorted && tid < nt) {
            const uint32_t gi = base + tid, c = L.rows[tid];
            for (uint32_t s = 1; s < c; s++) {
                const uint32_t tag = pj[size_t(s) * stride + gi];
                uint32_t q = s;
                if ((pj[size_t(s - 1) * stride + gi] & kIdxMask) < (tag & kIdxMask)) continue;
                const spring9 sp = ld_rec(ps + (size_t(s) * stride + gi) * kSpringRec);
                while (q > 0) {
                    const uint32_t prev = pj[size_t(q - 1) * stride + gi];
                    if ((prev & kIdxMask) < (tag & kIdxMask)) break;
                    pj[size_t(q) * stride + gi] = prev;
                    st_rec(ps + (size_t(q) * stride + gi) * kSpringRec,
                           ld_rec(ps + (size_t(q - 1) * stride + gi) * kSpringRec));
                    q--;
                }
                pj[size_t(q) * stride + gi] = tag;
                st_rec(ps + (size_t(q) * stride + gi) * kSpringRec, sp);
            }
        }
    if constexpr (W < 64) {
        if (tid < 6u * W) L.A[r0][i] = acct;
        __syncthreads();
    }
    if constexpr (FAC) {
        // the other set of facets for the next launch, moved by this step
        if (b.start == 0 && tid == kTileThreads - 1 && mode != TILE_FORCE) {
            const facet_dev *F = Vi.facets + size_t(b.slot) * Vi.max_facets;
            facet_dev *O = Vo.facets + size_t(b.slot) * Vo.max_facets;
            for (uint32_t f = 0; f < nf; f++) O[f] = F[f];
            if (Vi.facet_steps) advance_facets(O, int(nf), dt);
        }
    }
    // wavefront (or row) 0: force, velocity and position; 1: torque, angular
    // velocity and orientation
    if (r0 >= 2 || i >= nt) return;
    vec a;
    if constexpr (W == 64) a = accv;
    else a = vec{L.A[3 * r0][i], L.A[3 * r0 + 1][i], L.A[3 * r0 + 2][i]};
    if constexpr (FAC)
        if (nf) {
            fold_facets(0);
            a = a + fsum;
        }
    d3 a64;
    if constexpr (PREC == HG_PRECISION_FP64) a64 = a;
    else a64 = tod(a);
    if (mode != TILE_STEP) st3(r0 ? Vi.al : Vi.a, g, a64);
    if (mode == TILE_FORCE) return;
    d3 u = own(1 + int(r0), i);
    u = u + a64 * half;
    if (mode == TILE_STEP) {
        u = u + a64 * half;
        if (r0 == 0) st3(Vo.x, g, own(0, i) + u * dt);
        else st3(Vi.th, g, own(3, i) + u * dt);
    } else {
        if (r0 == 0) st3(Vo.x, g, own(0, i));
        if (nonfinite(u, u)) {
            atomicOr(&Vi.flags[FLAG_NUMERIC], 1);
            if (Vi.sflags) atomicOr(&Vi.sflags[b.slot], HG_FAULT_NUMERIC);
        }
    }
    st3(r0 ? Vo.w : Vo.v, g, u);
}

// The first kick and drift of an interval, from the systems' own buffers into
// Vo (the same buffers or the other set); the facets are copied along.
__global__ void __launch_bounds__(64) k_tile_kick(pool_view V, pool_view Vo, const wide_block *map, uint32_t width,
                                                  double half, double dt) {
    const wide_block b = tile_block(map, V, width);
    const uint32_t n = b.n & kIdxMask;
    if (Vo.facets != V.facets && b.start == 0 && threadIdx.x == 0) {
        const uint32_t nf = V.meta[b.slot].nf;
        for (uint32_t f = 0; f < nf; f++)
            Vo.facets[size_t(b.slot) * V.max_facets + f] = V.facets[size_t(b.slot) * V.max_facets + f];
    }
    if (threadIdx.x >= width || b.start + threadIdx.x >= n) return;
    const uint32_t g = b.offset + b.start + threadIdx.x;
    const d3 v = ld3(V.v, g) + ld3(V.a, g) * half, w = ld3(V.w, g) + ld3(V.al, g) * half;
    st3(Vo.x, g, ld3(V.x, g) + v * dt);
    st3(V.th, g, ld3(V.th, g) + w * dt);
    st3(Vo.v, g, v);
    st3(Vo.w, g, w);
}

}  // namespace
}  // namespace hg

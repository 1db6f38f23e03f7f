// One pair's functors for the kernels that spread pairs over threads
// (tile_step.h, the tiny-system kernel): the same expressions in the same order
// as the per-particle walk's pair_fold_vw, split into the parts that a pair
// needs.
#pragma once

#include "force_device.h"

namespace hg {

// Mixed: pair_fold_mx's.
template <int PREC>
struct prec_types {
    using term = double;
    using vec = d3;
};
template <>
struct prec_types<HG_PRECISION_MIXED> {
    using term = float;
    using vec = f3;
};

// hamaker_eval, lr_hamaker_eval and simplified_hamaker_eval of r = xj - xi,
// with the distance taken once.
template <int HAM>
__device__ __forceinline__ d3 hamaker_along(const hg_hamaker_params &p, double dist, d3 u) {
    if (HAM == HG_HAMAKER_NONE || (HAM == HG_HAMAKER_LIMITED && dist > p.r_cutoff)) return zero3();
    double h = dist - 2.0 * p.r_part;
    if (h < p.h0) h = p.h0;
    d3 f;
    if constexpr (HAM == HG_HAMAKER_SIMPLIFIED) f = 2.0 * p.A * p.r_part / sq(h) * u;
    else f = hamaker_scalar(p.A, p.r_part, h) * u;
    return f / p.mass;
}
template <int HAM>
__device__ __forceinline__ d3 hamaker_lin(const hg_hamaker_params &p, d3 r) {
    if constexpr (HAM == HG_HAMAKER_NONE) return zero3();
    const double z = dot(r, r), dist = sqrt(z);
    if (HAM == HG_HAMAKER_LIMITED && dist > p.r_cutoff) return zero3();
    return hamaker_along<HAM>(p, dist, z > 0.0 ? r / dist : r);
}

// The contact functor's overlap is 2 r minus a distance, a square root and three
// divisions away from the squared distance d2. Beyond the squared contact
// distance and a margin far above rounding it is negative; the margin is at
// least the smallest normal number, below which d2 has few bits, and an infinite
// d2, whose direction is zero or not a number, takes the functor's own course.
struct contact_reach {
    double d2_max;
    __device__ __forceinline__ explicit contact_reach(double r_part) {
        const double reach = 2.0 * r_part;
        d2_max = fmax(reach * reach * (1.0 + 1e-12), 0x1p-1022);
    }
    __device__ __forceinline__ bool beyond(double d2) const { return d2 > d2_max && d2 < __builtin_huge_val(); }
};

template <int HAM, int PREC>
struct pair_eval {
    using vec = typename prec_types<PREC>::vec;
    const hg_params &p;
    const mixed_consts &m;
    contact_reach reach;

    __device__ __forceinline__ pair_eval(const hg_params &P, const mixed_consts &M)
        : p(P), m(M), reach(P.contact.r_part) {}
    // A bonded pair: its term and new springs; true when the bond breaks
    // (this evaluation is still the bonded one).
    template <class NECK>
    __device__ __forceinline__ bool bonded(d3 xi, d3 vi, d3 wi, d3 xj, d3 vj, d3 wj, spring9 &sp, NECK &&neck,
                                           vec &lin, vec &ang) const {
        bool broke = false;
        if constexpr (PREC == HG_PRECISION_FP64) {
            d3 ftot;
            // the Hamaker term's direction is -n: one square root and three
            // divisions fewer, and the same bits but for the sign of a zero,
            // which the sum over the pairs does not keep
            const d3 d = xi - xj;
            const double z = dot(d, d), dist = sqrt(z);
            const d3 n = z > 0.0 ? d / dist : d;
            const acc6 b = sinter_eval_n(p.sinter, d, n, vi, vj, wi, wj, sp, ftot);
            if (p.sinter_breaking) broke = norm(ftot) > neck();
            lin = HAM != HG_HAMAKER_NONE ? b.lin + hamaker_along<HAM>(p.hamaker, dist, -n) : b.lin;
            ang = b.ang;
        } else {
            double dist;
            d3 n64;
            f3 n;
            pair_kinematics_mx(xi, xj, dist, n64, n);
            bool keep;
            const accf b = bonded_or_contact_mx<true>(
                m, dist, n64, n, vi, wi, [&](d3 &v, d3 &w) { v = vj, w = wj; }, sp, keep);
            if (m.s_breaking) broke = sqrtf(dotf(b.lin, b.lin)) * m.s_m > float(neck());
            f3 h = zerof();
            if constexpr (HAM != HG_HAMAKER_NONE) h = hamaker_mx<HAM>(m, dist, n);
            lin = b.lin + h;
            ang = b.ang;
        }
        return broke;
    }
    // The Hamaker term of an unbonded pair and, with CONTACT, whether the
    // pair is in contact.
    template <bool CONTACT>
    __device__ __forceinline__ bool free(d3 xi, d3 xj, vec &lin) const {
        bool touching = false;
        if constexpr (PREC == HG_PRECISION_FP64) {
            if constexpr (CONTACT) {
                const d3 d = xi - xj;
                if (!reach.beyond(dot(d, d))) {
                    const double overlap = 2.0 * p.contact.r_part - dot(d, normalized(d));
                    touching = !(overlap <= 0);
                }
            }
            lin = hamaker_lin<HAM>(p.hamaker, xj - xi);
        } else {
            const d3 d = xi - xj;
            const double d2 = dotm(d, d);
            lin = zerof();
            if (!(d2 > m.far2)) {
                double dist;
                d3 n64;
                f3 n;
                pair_kinematics_mx(xi, xj, dist, n64, n);
                if constexpr (CONTACT) touching = !(m.c_r2 - dist <= 0.0);
                if constexpr (HAM != HG_HAMAKER_NONE) lin = hamaker_mx<HAM>(m, dist, n);
            } else {
                if constexpr (HAM != HG_HAMAKER_NONE) lin = hamaker_far_mx<HAM>(m, d, d2);
            }
        }
        return touching;
    }
    // The contact functor of a touching pair (without its Hamaker term).
    __device__ __forceinline__ void contact(d3 xi, d3 vi, d3 wi, d3 xj, d3 vj, d3 wj, spring9 &sp, vec &lin,
                                            vec &ang) const {
        bool keep;
        auto vw = [&](d3 &v, d3 &w) { v = vj, w = wj; };
        if constexpr (PREC == HG_PRECISION_FP64) {
            const acc6 b = contact_eval_vw(p.contact, xi, xj, vi, wi, vw, sp, keep);
            lin = b.lin;
            ang = b.ang;
        } else {
            double dist;
            d3 n64;
            f3 n;
            pair_kinematics_mx(xi, xj, dist, n64, n);
            const accf b = bonded_or_contact_mx<false>(m, dist, n64, n, vi, wi, vw, sp, keep);
            lin = b.lin;
            ang = b.ang;
        }
    }
};

}  // namespace hg

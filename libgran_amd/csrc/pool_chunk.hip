// The chunk and tile kernels of one binary functor and pair mode; the Makefile
// compiles this file once for each (HG_BIN, HG_PAIRS), in parallel.
#include "tile_step.h"

namespace hg {

namespace {

template <int HAM, int PREC, bool FAC, int TPB>
hipError_t launch_chunk_k(const hg_params &p, const pool_view &V, const chunk_launch &c, hipStream_t s) {
    const auto kernel = &k_pool_chunk<HG_BIN, HAM, HG_PAIRS, PREC, FAC, TPB>;
    if (c.lds_cap > 0) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(c.lds_cap));
        if (e != hipSuccess) return e;
    }
    kernel<<<c.grid, TPB, c.lds_cap, s>>>(p, make_mixed_consts(p), V, c.order, c.packs, c.count, c.counter, c.nsteps,
                                          c.dt, c.lds_cap);
    return hipGetLastError();
}

template <int HAM>
hipError_t launch_chunk_h(const hg_params &p, const pool_view &V, const chunk_launch &c, hipStream_t s) {
#define HG_KCASE(PREC, FAC, TPB) \
    if (p.precision == PREC && c.facets == FAC && c.tpb == TPB) return launch_chunk_k<HAM, PREC, FAC, TPB>(p, V, c, s);
    HG_KCASE(HG_PRECISION_MIXED, true, 256)
    HG_KCASE(HG_PRECISION_MIXED, false, 256)
    HG_KCASE(HG_PRECISION_FP64, true, 256)
    HG_KCASE(HG_PRECISION_FP64, false, 256)
    HG_KCASE(HG_PRECISION_MIXED, true, 512)
    HG_KCASE(HG_PRECISION_MIXED, false, 512)
    HG_KCASE(HG_PRECISION_FP64, true, 512)
    HG_KCASE(HG_PRECISION_FP64, false, 512)
#undef HG_KCASE
    return hipErrorInvalidValue;
}

template <int HAM>
hipError_t launch_tile_h(const hg_params &p, const pool_view &Vi, const pool_view &Vo, const wide_block *map,
                         unsigned blocks, int mode, bool facets, double half, double dt, hipStream_t s) {
    const mixed_consts mc = make_mixed_consts(p);
    if constexpr (HG_PAIRS == HG_PAIRS_NEIGHBOR_LIST && HG_BIN != HG_BINARY_NONE)
        if (p.precision == HG_PRECISION_FP64 && !facets && blocks > kTwoOnEachCu) {
            k_tile_step<HG_BIN, HAM, HG_PAIRS, HG_PRECISION_FP64, false, 3>
                <<<blocks, kTileThreads, 0, s>>>(p, mc, Vi, Vo, map, mode, half, dt);
            return hipGetLastError();
        }
#define HG_KCASE(PREC, FAC)                                                       \
    if (p.precision == PREC && facets == FAC)                                     \
        k_tile_step<HG_BIN, HAM, HG_PAIRS, PREC, FAC>                             \
            <<<blocks, kTileThreads, 0, s>>>(p, mc, Vi, Vo, map, mode, half, dt);
    HG_KCASE(HG_PRECISION_MIXED, true)
    HG_KCASE(HG_PRECISION_MIXED, false)
    HG_KCASE(HG_PRECISION_FP64, true)
    HG_KCASE(HG_PRECISION_FP64, false)
#undef HG_KCASE
    return hipGetLastError();
}

}  // namespace

template <>
hipError_t launch_chunk_b<HG_BIN, HG_PAIRS>(const hg_params &p, const pool_view &V, const chunk_launch &c,
                                            hipStream_t s) {
    if (p.hamaker_model == HG_HAMAKER_NONE) return launch_chunk_h<HG_HAMAKER_NONE>(p, V, c, s);
    if (p.hamaker_model == HG_HAMAKER_FULL) return launch_chunk_h<HG_HAMAKER_FULL>(p, V, c, s);
    if (p.hamaker_model == HG_HAMAKER_LIMITED) return launch_chunk_h<HG_HAMAKER_LIMITED>(p, V, c, s);
    if (p.hamaker_model == HG_HAMAKER_SIMPLIFIED) return launch_chunk_h<HG_HAMAKER_SIMPLIFIED>(p, V, c, s);
    return hipErrorInvalidValue;
}

template <>
hipError_t launch_tile_b<HG_BIN, HG_PAIRS>(const hg_params &p, const pool_view &Vi, const pool_view &Vo,
                                           const wide_block *map, unsigned blocks, int mode, bool facets, double half,
                                           double dt, hipStream_t s) {
    if (blocks == 0) return hipSuccess;
#define HG_TCASE(H) \
    if (p.hamaker_model == H) return launch_tile_h<H>(p, Vi, Vo, map, blocks, mode, facets, half, dt, s);
    HG_TCASE(HG_HAMAKER_NONE)
    HG_TCASE(HG_HAMAKER_FULL)
    HG_TCASE(HG_HAMAKER_LIMITED)
    HG_TCASE(HG_HAMAKER_SIMPLIFIED)
#undef HG_TCASE
    return hipErrorInvalidValue;
}

#if HG_PAIRS == 0
static_assert(HG_PAIRS_ALL == 0, "the walk is all pairs'");
template <>
hipError_t launch_walk_b<HG_BIN>(const hg_params &p, const pool_view &V, const wide_block *map, unsigned blocks,
                                 int pass, hipStream_t s) {
    if (blocks == 0) return hipSuccess;
    const mixed_consts mc = make_mixed_consts(p);
#define HG_WCASE(H, PREC)                                                                  \
    if (p.hamaker_model == H && p.precision == PREC) {                                     \
        k_walk_force<HG_BIN, H, PREC><<<blocks, kWalkBlock, 0, s>>>(p, mc, V, map, pass);  \
        return hipGetLastError();                                                          \
    }
    HG_WCASE(HG_HAMAKER_NONE, HG_PRECISION_FP64)
    HG_WCASE(HG_HAMAKER_FULL, HG_PRECISION_FP64)
    HG_WCASE(HG_HAMAKER_LIMITED, HG_PRECISION_FP64)
    HG_WCASE(HG_HAMAKER_SIMPLIFIED, HG_PRECISION_FP64)
    HG_WCASE(HG_HAMAKER_NONE, HG_PRECISION_MIXED)
    HG_WCASE(HG_HAMAKER_FULL, HG_PRECISION_MIXED)
    HG_WCASE(HG_HAMAKER_LIMITED, HG_PRECISION_MIXED)
    HG_WCASE(HG_HAMAKER_SIMPLIFIED, HG_PRECISION_MIXED)
#undef HG_WCASE
    return hipErrorInvalidValue;
}
#endif

}  // namespace hg

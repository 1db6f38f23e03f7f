// How the tiles (tile_step.h) look up entries of their pair-state rows. Plain
// functions, compiled for the device by the kernels and for the host by the
// tests.
#pragma once

#include <stdint.h>

#if defined(__HIP__)
#define HG_ROW __host__ __device__ __forceinline__
#else
#define HG_ROW inline
#endif

namespace hg {

// Pair-state table entry tag: bit 31 marks a bonded (alt_sinter) pair; the low
// 31 bits are the partner index j.
constexpr uint32_t kBondBit = 0x80000000u;
constexpr uint32_t kIdxMask = 0x7fffffffu;
constexpr uint32_t kNoEntry = 0xffffffffu;  // (kNoEntry & kIdxMask) exceeds every valid j

constexpr uint32_t kNoRowSlot = 0xFFFu;

// The slot of partner j in a row of `count` entries, tag(s) the tag of slot s.
// It is the first match: removing ended entries leaves their old tags beyond
// the row's end, and a slot there that another thread has claimed (`count`
// includes it) holds such a tag, j's own perhaps, until the claimer has written
// its own.
template <class TAG>
HG_ROW uint32_t row_slot(uint32_t count, uint32_t j, TAG &&tag) {
    for (uint32_t s = 0; s < count; s++)
        if ((tag(s) & kIdxMask) == j) return s;
    return kNoRowSlot;
}

}  // namespace hg

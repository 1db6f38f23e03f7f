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

// A queued pair's place: its list position among those the tile takes at a time
// and its particle (position * width + particle, at most kTilePlaces) and its
// slot in the particle's row. A row holds distinct partners, so a slot of 22
// bits is beyond what the tables of such a system would fit in memory.
constexpr uint32_t kPlaceBits = 10, kTilePlaces = 1u << kPlaceBits;
constexpr uint32_t kNoRowSlot = ~0u >> kPlaceBits;
HG_ROW uint32_t queue_word(uint32_t place, uint32_t slot) { return place | (slot << kPlaceBits); }
HG_ROW uint32_t queue_place(uint32_t word) { return word & (kTilePlaces - 1u); }
HG_ROW uint32_t queue_slot(uint32_t word) { return word >> kPlaceBits; }

// The slot of partner j in a row of `count` entries, tag(s) the tag of slot s.
// It is the first match: removing ended entries leaves old tags beyond the
// row's end, and a slot there that another thread has claimed, should `count`
// include it, holds such a tag, j's own perhaps, until the claimer has written
// its own.
template <class TAG>
HG_ROW uint32_t row_slot(uint32_t count, uint32_t j, TAG &&tag) {
    for (uint32_t s = 0; s < count; s++)
        if ((tag(s) & kIdxMask) == j) return s;
    return kNoRowSlot;
}

}  // namespace hg

// bins.hpp - where binned mode keeps a bin's entries, and the order in which
// a wave stores them: plain functions that the kernels (raster.hip) and a host
// test share.
#pragma once
#include <cstdint>
#include "axr_math.hpp"

namespace axr {

// Bins of binned mode: level k of a bin holds 2^(bin0_shift + k) entries, so
// BIN_LEVELS levels reach 2^31 entries for the smallest first level.
constexpr uint32_t BIN0_LEAN_SHIFT = 4, BIN0_MIN_SHIFT = 5, BIN0_MAX_SHIFT = 12;
constexpr uint32_t COUNT_BLOCK = 8192;         // words of tile_count that bins are spread over
constexpr uint32_t BIN_LEVELS = 27;
constexpr uint32_t CHUNK_NONE = 0xFFFFFFFFu;   // a level the pools had no room for

// The word of tile_count that counts bin t's entries.  Atomics on one cache
// line wait for each other (~9 ns each, whatever word they name: 7M spread
// over 3,600 neighbouring words take 530 us, over twice the lines 290), and a
// mesh fills neighbouring bins at the same time, so a block of 8,192 words
// holds its bins in runs of four, each run in another of its 256 lines.  The
// runs are there for triangles over two or three bins, whose atomics on one
// line travel together (the 4M-triangle soup's k_setup 255 us, 279 with every
// bin in another line).  k_setup of 40 mixed views 88 -> 69 us, of a 150k soup
// 25 -> 19.5, of the 1M-triangle frame 20.7 -> 18.
AXR_HD uint32_t count_word(uint32_t t) {
    return (t & ~(COUNT_BLOCK - 1u)) | ((t & 0x3FCu) << 3) | (t & 3u) | ((t >> 8) & 28u);
}

// Where a bin's entry `slot` lies: entry `offset` of level `level`.
struct BinSlot {
    uint32_t level, offset;
};
AXR_HD BinSlot bin_slot(uint32_t bin0_shift, uint32_t slot) {
    const uint32_t level = 31u - (uint32_t)__builtin_clz((slot >> bin0_shift) + 1u);
    return BinSlot{level, slot - (((1u << level) - 1u) << bin0_shift)};
}

// Stores the Q entries per lane whose slots a wave has taken, waves against
// waves: s.near(q) stores entry q if it lies in its bin's first level, else
// returns true; where the wave has such entries (s.any), s.open(q) publishes
// the level that entry q opens, if it does, and waits for nothing, and
// s.fill(q) stores entry q, after waiting for its level if another lane opens
// that.  Every open comes before every fill: a wave that waited with a level
// of its own unpublished could wait for a wave that waits for that level (the
// slots are taken by atomics on different words, in flight together, so either
// wave may be the first on one word and the second on the other).
template <uint32_t Q, class Store>
AXR_HD void place_entries(Store& s) {
    bool far = false;
#pragma unroll
    for (uint32_t q = 0; q < Q; ++q) far |= s.near(q);
    if (!s.any(far)) return;
#pragma unroll
    for (uint32_t q = 0; q < Q; ++q) s.open(q);
#pragma unroll
    for (uint32_t q = 0; q < Q; ++q) s.fill(q);
}

}  // namespace axr

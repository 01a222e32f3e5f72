// tile_plan.h - which frames may have their tile lists binned, and the integers that
// a binned frame's projection carries. Plain C++ without HIP, so that the rules are
// checked on the host (tests/tile_plan_check.cpp).
#pragma once

#include <stdint.h>

namespace gs {

constexpr int kBinnedTiles = 1 << 14;  // most tiles of a binned frame (32 KB of LDS counters)

// A binned frame's compaction look-back carries the visible count and the candidate
// total in one 62-bit value: the count above, the candidates below. The total is only
// known after that scan and nothing saturates on the way, so a frame is binned only if
// its fields hold every total that its sizes allow (binned_fits): N Gaussians that
// each cover all T tiles.
constexpr int kBinnedCandBits = 34, kBinnedCountBits = 28;
static_assert(kBinnedCandBits + kBinnedCountBits <= 62, "the look-back's value has 62 bits");

constexpr uint64_t binned_pack(uint32_t count, uint64_t cands) {
    return ((uint64_t)count << kBinnedCandBits) | cands;
}
constexpr uint64_t binned_count(uint64_t v) { return v >> kBinnedCandBits; }
constexpr uint64_t binned_cands(uint64_t v) { return v & ((1ull << kBinnedCandBits) - 1); }

// Whether the counts of a frame of n Gaussians and `tiles` tiles fit those fields, its
// tiles the counters in LDS.
constexpr bool binned_fits(int64_t n, int64_t tiles) {
    return tiles <= kBinnedTiles && n < ((int64_t)1 << kBinnedCountBits) &&
           (uint64_t)n * (uint64_t)tiles < (1ull << kBinnedCandBits);
}

}  // namespace gs

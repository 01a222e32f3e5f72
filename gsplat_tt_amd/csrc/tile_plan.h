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

// How frames make their tile lists, from what the finished frames of the same sizes
// found. Binning (launch_binned_lists) needs no depth sort and fewer launches but stores
// each pair at its list's end and sorts each list on its own, so it wins up to about
// 2.4M pairs (us a frame alone and in a path, blocks against binned; 1280x720: 1.1M
// pairs 317, 213 / 243, 186; 1.7M 366, 246 / 294, 227; 2.8M 434, 295 / 380, 291;
// 1237x822: 1.5M 263, 173 / 201, 156; 3.0M 314, 221 / 320, 255; 5.0M 367, 276 / 477,
// 407; 400x300, 3100 pairs a tile: 1.5M 283, 234 / 294, 186). The pairs of a view are
// not known before it is rendered: frames start from the number of Gaussians and go
// on with the pairs of the frames that finished, with a gap between the two limits so
// that a camera path does not alternate.
// What was found is kept for several sizes (a trainer's photographs, a thumbnail beside
// the full view), frames and training forwards apart, the least recently used given up.
// A scene set anew with as many Gaussians goes on from what the last one found: a wrong
// start costs time in one frame, never a result.
class TilePlans {
public:
    enum Kind { kFrame, kTrain };
    // Whether the next frame of these sizes is binned.
    bool binned(Kind kind, int64_t n, int64_t tiles) {
        return entry(kind, n, tiles).binned && binned_fits(n, tiles);
    }
    // A frame of these sizes has finished with `pairs` pairs.
    void seen(Kind kind, int64_t n, int64_t tiles, int64_t pairs) {
        Entry& e = entry(kind, n, tiles);
        if (pairs > kMost) e.binned = false;
        if (pairs < kAgain) e.binned = true;
    }

    static constexpr int kEntries = 16;
    static constexpr int64_t kFirst = 1 << 20, kMost = 2400000, kAgain = 1800000;

private:
    struct Entry {
        Kind kind = kFrame;
        int64_t n = -1, tiles = -1;
        uint64_t used = 0;
        bool binned = false;
    };
    Entry& entry(Kind kind, int64_t n, int64_t tiles) {
        Entry* at = &e_[0];
        for (Entry& e : e_) {
            if (e.n == n && e.tiles == tiles && e.kind == kind) {
                e.used = ++clock_;
                return e;
            }
            if (e.used < at->used) at = &e;
        }
        *at = Entry{kind, n, tiles, ++clock_, n <= kFirst};
        return *at;
    }
    Entry e_[kEntries];
    uint64_t clock_ = 0;
};

}  // namespace gs

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

// Most candidates of a binned frame, for which its buffers are sized: the bins take a word
// per two tiles and 2048 of them (64 MB at 2^14 tiles; for a context's whole pair
// capacity, which only grows, gigabytes). Views with 2.4M pairs have 2.5M to 3M of them. A
// frame that has more is made again another way, which takes no longer there.
constexpr uint32_t kBinnedCands = 1u << 22;

// How frames make their tile lists, from what the finished frames of the same sizes
// found. Binning (launch_binned_lists) needs no depth sort and fewer launches but stores
// each pair at its list's end and sorts each list on its own, so it wins up to about
// 2.4M pairs (us a frame alone and in a path, blocks against binned; 1280x720: 1.1M
// pairs 317, 213 / 243, 186; 1.7M 366, 246 / 294, 227; 2.8M 434, 295 / 380, 291;
// 1237x822: 1.5M 263, 173 / 201, 156; 3.0M 314, 221 / 320, 255; 5.0M 367, 276 / 477,
// 407; 400x300, 3100 pairs a tile: 1.5M 283, 234 / 294, 186). A list past two runs of 2048
// is searched run by run in all its others, while the other ways take as long however
// the pairs lie: every run past two of the longest list costs a frame 6 us, as 0.3M
// pairs do (binned against pairs sorted by tile, the longest list in brackets: 320x240
// 0.44M pairs [9.4K] 168, 100 / 204, 122; 640x480 in tiles of 32 0.99M [7.3K] 189, 127 /
// 229, 149; 320x240 0.87M [19K] 248, 143 / 250, 146; 640x480 in tiles of 32 1.14M [25K]
// 325, 195 / 291, 194; 160x120 in tiles of 32 0.48M [64K] 749, 301 / 599, 259; one tile
// 0.05M 790, 216 / 708, 198 and 1M 4082, 1607 / 635, 224).
// The lists of a view are not known before it is rendered: the first frame goes by the
// number of Gaussians, later ones by the lists of the frames that finished, with a gap
// between the two limits so that a camera path does not alternate.
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
    // A frame of these sizes has finished: it had `cands` candidates, of which `pairs` are
    // left, `longest` in one tile.
    void seen(Kind kind, int64_t n, int64_t tiles, int64_t cands, int64_t pairs,
              int64_t longest) {
        Entry& e = entry(kind, n, tiles);
        const int64_t c = cost(pairs, longest);
        if (c > kMost || cands > kBinnedCands) e.binned = false;
        if ((c < kAgain && cands < kBinnedCands / 4 * 3) ||
            (!e.known && c <= kMost && cands <= kBinnedCands))
            e.binned = true;
        e.known = true;
    }
    // A binned frame of these sizes did not fit kBinnedCands: it is made again, not binned.
    void past(Kind kind, int64_t n, int64_t tiles) { entry(kind, n, tiles).binned = false; }

    static constexpr int kEntries = 16;
    // (2 pairs a Gaussian reach kMost: 0.6 to 5 in the views measured)
    static constexpr int64_t kFirst = 1 << 20, kMost = 2400000, kAgain = 1800000;

private:
    // In pairs: those there are, and what merging the longest list takes.
    static constexpr int64_t cost(int64_t pairs, int64_t longest) {
        return pairs + 150 * (longest > 4096 ? longest - 4096 : 0);
    }
    // A size not seen before: two pairs a Gaussian, four times the mean in one tile.
    static constexpr bool first(int64_t n, int64_t tiles) {
        return n <= kFirst && cost(2 * n, 4 * n / (tiles > 0 ? tiles : 1)) <= kMost;
    }
    struct Entry {
        Kind kind = kFrame;
        int64_t n = -1, tiles = -1;
        uint64_t used = 0;
        bool binned = false;
        bool known = false;  // a frame has finished
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
        *at = Entry{kind, n, tiles, ++clock_, first(n, tiles), false};
        return *at;
    }
    Entry e_[kEntries];
    uint64_t clock_ = 0;
};

}  // namespace gs

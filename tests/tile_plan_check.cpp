// Host-only checks of the tile-list rules (gsplat_tt_amd/csrc/tile_plan.h), built with
// g++ by tests/test_tile_plan.py.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "tile_plan.h"

static int fails = 0;
#define CHECK(c)                                                              \
    do {                                                                      \
        if (!(c)) {                                                           \
            std::fprintf(stderr, "FAIL line %d: %s\n", __LINE__, #c);         \
            ++fails;                                                          \
        }                                                                     \
    } while (0)

// The compaction's sums over partitions of `part` Gaussians that each cover every
// tile, as the look-back forms them: what the last partition reports must be the
// count and the total, and the flag bits above must stay free.
static void full_cover(int64_t n, int64_t tiles, int64_t part) {
    uint64_t v = 0;
    for (int64_t at = 0; at < n; at += part) {
        const int64_t c = n - at < part ? n - at : part;
        v += gs::binned_pack((uint32_t)c, (uint64_t)c * (uint64_t)tiles);
    }
    CHECK(gs::binned_count(v) == (uint64_t)n);
    CHECK(gs::binned_cands(v) == (uint64_t)n * (uint64_t)tiles);
    CHECK((v >> 62) == 0);
}

static void fields() {
    const int64_t most = gs::kBinnedTiles;
    // one Gaussian fewer than 2^34 candidates fits, 2^34 does not (and a first frame of
    // 2^20 Gaussians over 2^14 tiles is exactly that)
    CHECK(gs::binned_fits((1 << 20) - 1, most));
    CHECK(!gs::binned_fits(1 << 20, most));
    CHECK(!gs::binned_fits(4000000, most));
    CHECK(gs::binned_fits(4000000, 4000));
    CHECK(!gs::binned_fits(1, most + 1));
    CHECK(!gs::binned_fits((int64_t)1 << 28, 1));
    CHECK(gs::binned_fits(((int64_t)1 << 28) - 1, 1));
    for (const int64_t n : {1ll, 511ll, 513ll, 1ll << 18, (1ll << 20) - 1, 1ll << 20, 1ll << 22,
                            6000000ll, (1ll << 28) - 1, 1ll << 28})
        for (const int64_t t : {1ll, 63ll, 64ll, 65ll, 3600ll, 16383ll, 16384ll, 16385ll})
            if (gs::binned_fits(n, t)) full_cover(n, t, n > (1 << 18) ? 2048 : 512);
}

// Sizes that alternate keep what each of them found, up to as many as are remembered.
static void sizes() {
    using P = gs::TilePlans;
    const int64_t n = 1000000, full = 3600, thumb = 300;
    {
        P p;  // few Gaussians start binned, many do not
        CHECK(p.binned(P::kFrame, P::kFirst, full) && !p.binned(P::kFrame, P::kFirst + 1, full));
        CHECK(!p.binned(P::kFrame, 1000, gs::kBinnedTiles + 1));
    }
    {
        P p;
        for (int k = 0; k < 4; ++k) {
            p.binned(P::kFrame, n, full);
            p.seen(P::kFrame, n, full, 5000000, 5000000, 3000);
            p.binned(P::kFrame, n, thumb);
            p.seen(P::kFrame, n, thumb, 700000, 700000, 4096);
            CHECK(!p.binned(P::kFrame, n, full) && p.binned(P::kFrame, n, thumb));
            CHECK(p.binned(P::kTrain, n, full));  // a training forward's pairs are its own
        }
        p.seen(P::kFrame, n, full, P::kAgain, P::kAgain, 0);  // between the limits: as it was
        CHECK(!p.binned(P::kFrame, n, full));
        p.seen(P::kFrame, n, full, P::kAgain - 1, P::kAgain - 1, 0);
        CHECK(p.binned(P::kFrame, n, full));
        p.seen(P::kFrame, n, full, P::kMost, P::kMost, 0);
        CHECK(p.binned(P::kFrame, n, full));
    }
    {
        P p;  // many Gaussians, few pairs: binned from the second frame, also between others
        for (int k = 0; k < P::kEntries; ++k) {
            CHECK(!p.binned(P::kFrame, 3000000, 100 + k));
            p.seen(P::kFrame, 3000000, 100 + k, 500000, 500000, 0);
        }
        for (int k = 0; k < P::kEntries; ++k) CHECK(p.binned(P::kFrame, 3000000, 100 + k));
        CHECK(!p.binned(P::kFrame, 3000000, 99));  // one more size: the oldest is given up
        CHECK(p.binned(P::kFrame, 3000000, 100 + P::kEntries - 1));
        CHECK(!p.binned(P::kFrame, 3000000, 100));
    }
}

// A frame of few pairs in long lists is not binned, however few tiles it has or how its
// pairs spread over the others.
static void lists() {
    using P = gs::TilePlans;
    {   // the first frame that finishes decides by the upper limit, whatever was guessed
        P q;
        CHECK(!q.binned(P::kFrame, 300000, 70) && !q.binned(P::kFrame, 3000000, 3600));
        q.seen(P::kFrame, 300000, 70, 414000, 414000, 14914);  // 2.04M
        q.seen(P::kFrame, 3000000, 3600, P::kMost, P::kMost, 0);
        CHECK(q.binned(P::kFrame, 300000, 70) && q.binned(P::kFrame, 3000000, 3600));
    }
    P p;
    p.seen(P::kFrame, 100000, 3600, 500000, 500000, 4096);
    CHECK(p.binned(P::kFrame, 100000, 3600));
    p.seen(P::kFrame, 100000, 3600, 500000, 500000, 18000);  // 2.59M
    CHECK(!p.binned(P::kFrame, 100000, 3600));
    p.seen(P::kFrame, 100000, 3600, 500000, 500000, 14000);  // 1.99M: as it was
    CHECK(!p.binned(P::kFrame, 100000, 3600));
    p.seen(P::kFrame, 100000, 3600, 500000, 500000, 12000);  // 1.69M
    CHECK(p.binned(P::kFrame, 100000, 3600));
    p.seen(P::kFrame, 100000, 3600, 500000, 500000, 16000);  // 2.29M: as it was
    CHECK(p.binned(P::kFrame, 100000, 3600));
    // first frames: a scene over a few tiles has long lists, over many it has not
    CHECK(!p.binned(P::kFrame, 1 << 20, 1) && !p.binned(P::kFrame, 1 << 20, 63));
    CHECK(!p.binned(P::kFrame, 50000, 1) && p.binned(P::kFrame, 1000, 1));
    CHECK(p.binned(P::kFrame, 1000000, 3600) && p.binned(P::kFrame, 100000, 300));
}

// A frame of more candidates than a binned one has room for is not binned, and the bins
// stay small whatever the pair capacity is.
static void room() {
    using P = gs::TilePlans;
    const int64_t most = gs::kBinnedCands, pairs = 1000000;
    P p;
    CHECK(p.binned(P::kFrame, 500000, 3600));
    p.past(P::kFrame, 500000, 3600);
    CHECK(!p.binned(P::kFrame, 500000, 3600));
    p.seen(P::kFrame, 500000, 3600, most + 1, pairs, 0);
    CHECK(!p.binned(P::kFrame, 500000, 3600));
    p.seen(P::kFrame, 500000, 3600, most, pairs, 0);  // near its room: as it was
    CHECK(!p.binned(P::kFrame, 500000, 3600));
    p.seen(P::kFrame, 500000, 3600, most / 2, pairs, 0);
    CHECK(p.binned(P::kFrame, 500000, 3600));
    p.seen(P::kFrame, 500000, 3600, most, pairs, 0);
    CHECK(p.binned(P::kFrame, 500000, 3600));
    p.seen(P::kFrame, 500000, 3600, most + 1, pairs, 0);
    CHECK(!p.binned(P::kFrame, 500000, 3600));
    // a first frame that was not binned and had too many
    p.seen(P::kFrame, 3000000, 3600, most + 1, pairs, 0);
    CHECK(!p.binned(P::kFrame, 3000000, 3600));
}

int main() {
    fields();
    room();
    sizes();
    lists();
    if (fails == 0) std::puts("ok");
    return fails ? 1 : 0;
}

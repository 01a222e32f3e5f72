// Host-only checks of the shared host work (gsplat_tt_amd/csrc/host_threads.h), built
// with g++ by tests/test_host_threads.py: every byte copied once and every index
// visited once, with all the threads asked for, with some and with none.
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <system_error>
#include <thread>
#include <vector>

#include "host_threads.h"

static int fails = 0;
#define CHECK(c)                                                              \
    do {                                                                      \
        if (!(c)) {                                                           \
            std::fprintf(stderr, "FAIL line %d: %s\n", __LINE__, #c);         \
            ++fails;                                                          \
        }                                                                     \
    } while (0)

// A thread that cannot be made once `allowed` of them exist.
static int allowed = 0, made = 0;
struct LimitedThread {
    std::thread t;
    template <class F>
    explicit LimitedThread(F&& f) {
        if (made >= allowed)
            throw std::system_error(std::make_error_code(
                std::errc::resource_unavailable_try_again));
        ++made;
        t = std::thread(std::forward<F>(f));
    }
    LimitedThread(LimitedThread&&) = default;
    void join() { t.join(); }
};

static void copies(int workers, int limit, bool down) {
    allowed = limit;
    made = 0;
    const size_t sizes[3][5] = {{12, 12, 16, 4, 36}, {0, 1, 63, 64, 65}, {100000, 7, 0, 4097, 300001}};
    gs::ChunkCopyOf<LimitedThread> copy(workers, down);
    for (int c = 0; c < 12; ++c) {
        const size_t* sz = sizes[c % 3];
        size_t total = 0;
        for (int q = 0; q < 5; ++q) total += sz[q];
        std::vector<char> pin(total), host(total), want(total);
        for (size_t i = 0; i < total; ++i) want[i] = (char)(i * 7 + c);
        (down ? pin : host) = want;
        std::array<gs::Piece, 5> p;
        size_t off = 0;
        for (int q = 0; q < 5; ++q) {
            p[q] = {host.data() + off, off, sz[q]};
            off += sz[q];
        }
        copy.chunk(pin.data(), p);
        CHECK((down ? host : pin) == want);
    }
    CHECK(made == std::min(limit, std::max(workers, 1) - 1));
}

static void ranges(int64_t n, int limit) {
    allowed = limit;
    made = 0;
    std::vector<std::atomic<uint8_t>> seen((size_t)n);
    gs::parallel_for<LimitedThread>(n, [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) seen[(size_t)i].fetch_add(1);
    });
    bool once = true;
    for (auto& s : seen) once = once && s.load() == 1;
    CHECK(once);
}

int main() {
    for (const int workers : {1, 2, 3, 8})
        for (const int limit : {0, 1, 3, 100})
            for (const bool down : {false, true}) copies(workers, limit, down);
    { gs::ChunkCopy idle(4, true); }  // no chunk at all
    for (const int64_t n : {0ll, 1ll, 65536ll, 131072ll, 131073ll, 700001ll})
        for (const int limit : {0, 1, 100}) ranges(n, limit);
    CHECK(gs::host_threads(0) == 1 && gs::host_threads(1) == 1);
    CHECK(gs::host_threads(1 << 20) == (int)std::max(1u, std::thread::hardware_concurrency()));
    if (fails == 0) std::puts("ok");
    return fails ? 1 : 0;
}

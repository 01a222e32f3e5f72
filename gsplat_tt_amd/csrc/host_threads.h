// host_threads.h - host work shared by a few threads of one call. Plain C++ without
// HIP (tests/host_threads_check.cpp). A thread that cannot be made is not an error: the
// threads that there are, the calling one at least, do all of the work.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace gs {

// Threads for work that pays for at most `most` of them.
inline int host_threads(int64_t most) {
    if (most <= 1) return 1;
    const int64_t hw = std::max(1u, std::thread::hardware_concurrency());
    return (int)std::min(hw, most);
}

// f(lo, hi) over [0, n) in up to one range per 65536 elements; f must not throw.
template <class Thread = std::thread, class F>
void parallel_for(int64_t n, F&& f) {
    const int64_t workers = host_threads(n / 65536);
    if (workers <= 1) {
        f(0, n);
        return;
    }
    const int64_t chunk = (n + workers - 1) / workers;
    std::vector<Thread> ts;
    int64_t lo = chunk;  // the calling thread takes the first range
    try {
        ts.reserve((size_t)workers);
        for (; lo < n; lo += chunk) {
            const int64_t hi = std::min(n, lo + chunk);
            ts.emplace_back([&f, lo, hi] { f(lo, hi); });
        }
    } catch (const std::exception&) {
    }
    f(0, chunk);
    if (lo < n) f(lo, n);
    for (auto& t : ts) t.join();
}

// Threads that copy each announced chunk together with the calling one. A chunk is five
// arrays one after the other in a staging slot, each with its place in the caller's
// memory. Between chunks a worker gives up its turns for kAwake, about the transfer of
// one 8 MB slot, and then sleeps: woken for each chunk, a read of one slot took 385 us
// for 340.
struct Piece {
    char* host;
    size_t off, bytes;
};
template <class Thread = std::thread>
class ChunkCopyOf {
public:
    // workers: threads that copy, the calling one among them; down: out of the slot
    ChunkCopyOf(int workers, bool down) : down_(down) {
        try {
            ts_.reserve((size_t)std::max(workers, 1));
            for (int i = 1; i < workers; ++i) ts_.emplace_back([this, i] { work(i); });
        } catch (const std::exception&) {
        }
        w_ = (int)ts_.size() + 1;  // read by a worker after its first chunk is announced
    }
    ~ChunkCopyOf() {
        announce(true);
        for (auto& t : ts_) t.join();
    }
    ChunkCopyOf(const ChunkCopyOf&) = delete;
    ChunkCopyOf& operator=(const ChunkCopyOf&) = delete;

    // Copies a chunk at `pin`; returns when all of it is copied.
    void chunk(char* pin, const std::array<Piece, 5>& p) {
        pin_ = pin;
        p_ = p;
        left_.store(w_ - 1, std::memory_order_relaxed);
        announce(false);
        share(0);
        while (left_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
    }

private:
    void announce(bool stop) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            stop_ = stop;
            seq_.fetch_add(1, std::memory_order_release);
        }
        go_.notify_all();
    }
    void share(int i) const {
        for (const Piece& q : p_) {
            const size_t lo = q.bytes * (size_t)i / (size_t)w_ & ~size_t(63);
            const size_t hi = i + 1 == w_ ? q.bytes
                                          : q.bytes * (size_t)(i + 1) / (size_t)w_ & ~size_t(63);
            if (hi == lo) continue;
            if (down_) std::memcpy(q.host + lo, pin_ + q.off + lo, hi - lo);
            else std::memcpy(pin_ + q.off + lo, q.host + lo, hi - lo);
        }
    }
    static constexpr std::chrono::microseconds kAwake{250};
    void work(int i) {
        for (uint64_t seen = 0;; ++seen) {
            const auto until = std::chrono::steady_clock::now() + kAwake;
            while (seq_.load(std::memory_order_acquire) == seen &&
                   std::chrono::steady_clock::now() < until)
                std::this_thread::yield();
            {
                std::unique_lock<std::mutex> lock(mu_);
                go_.wait(lock, [&] { return seq_ != seen; });
                if (stop_) return;
            }
            share(i);
            left_.fetch_sub(1, std::memory_order_release);
        }
    }
    const bool down_;
    int w_ = 1;
    std::vector<Thread> ts_;
    std::mutex mu_;
    std::condition_variable go_;
    bool stop_ = false;
    std::atomic<uint64_t> seq_{0};  // announced chunks, and the stop
    std::atomic<int> left_{0};
    char* pin_ = nullptr;
    std::array<Piece, 5> p_{};
};
using ChunkCopy = ChunkCopyOf<>;

}  // namespace gs

// Host threads that move the chunks of one copy between pageable memory and
// pinned slots while the DMA of other chunks runs.
#pragma once
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstddef>
#include <thread>
#include <vector>

namespace mcmb {

// One turn of a wait for a counter of another thread.  The chunks of a copy
// follow each other within some 100 us, over which a sleep is too coarse (19 MB
// out took 90 us longer with sleeps from 100 us on): for the first 2 ms a turn
// yields.  A wait past them is for something else (the device's earlier work,
// say), which a process must not spend nine cores on: turns then sleep, for an
// eighth of the time waited so far and at most 1 ms.
class Backoff {
    const std::chrono::steady_clock::time_point t0 = std::chrono::steady_clock::now();

  public:
    void pause() const
    {
        using namespace std::chrono;
        const auto w = steady_clock::now() - t0;
        if (w < milliseconds(2)) std::this_thread::yield();
        else std::this_thread::sleep_for(std::min<steady_clock::duration>(w / 8, milliseconds(1)));
    }
};

// n threads for the nk chunks of a copy: move(t, k) moves thread t's stripe of
// chunk k.  The owner announces chunks by raising `ready`; the threads live for
// the whole copy, and progress is two counters, so no thread waits for a lock.
struct ChunkCrew {
    const int nth;
    std::vector<std::atomic<int>> done;   // threads that have moved chunk k
    std::atomic<long> ready{0};           // chunks the threads may move
    std::atomic<bool> stop{false};
    std::vector<std::thread> th;

    template <class F> ChunkCrew(int n, size_t nk, F move) : nth(n), done(nk)
    {
        for (auto& d : done) d.store(0, std::memory_order_relaxed);
        th.reserve(n);
        try {
            for (int t = 0; t < n; ++t)
                th.emplace_back([this, t, nk, move] {
                    for (size_t k = 0; k < nk; ++k) {
                        for (Backoff b; ready.load(std::memory_order_acquire) <= (long)k; b.pause())
                            if (stop.load(std::memory_order_relaxed)) return;
                        move(t, k);
                        done[k].fetch_add(1, std::memory_order_release);
                    }
                });
        } catch (...) {   // no further thread to be had
            join();
            throw;
        }
    }
    void join()
    {
        stop.store(true);
        for (auto& x : th) x.join();
    }
    void wait(size_t k) const
    {
        for (Backoff b; done[k].load(std::memory_order_acquire) < nth;) b.pause();
    }
    ~ChunkCrew() { join(); }
};

}  // namespace mcmb

// Threads that share a copy between host arrays.  Plain C++, so that the tests
// compile it alone.
#pragma once

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace st {

// The helper threads of a context's host transfers, made at its first large
// one and joined with it.  They share each piece with the calling thread.  The
// pieces of a transfer follow each other within some tens of microseconds, so
// after one they poll for the next; but a transfer may also wait for all the
// work enqueued before it, so they poll for SPIN at most and then sleep until a
// piece is there.  Threads that cannot be had are done without.
class Copiers {
public:
    Copiers()
    {
        const int hw = (int)std::thread::hardware_concurrency();
        const int n = hw - 1 < 0 ? 0 : hw - 1 < MOST ? hw - 1 : MOST;
        try {
            for (; have < n; have++) t[have] = std::thread([this, k = have] { work(k + 1); });
        } catch (const std::exception &) {
        }
    }
    ~Copiers()
    {
        stop.store(true);
        rouse();
        for (int k = 0; k < have; k++) t[k].join();
    }
    Copiers(const Copiers &) = delete;
    Copiers &operator=(const Copiers &) = delete;
    // a piece will come soon: sleeping threads poll for it
    void wake()
    {
        calls.fetch_add(1);
        rouse();
    }
    void copy(void *d, const void *s, size_t n)
    {
        dst = (char *)d;
        src = (const char *)s;
        size = n;
        left.store(have, std::memory_order_relaxed);
        turn.fetch_add(1);
        rouse();
        part(0);
        while (left.load(std::memory_order_acquire) > 0) std::this_thread::yield();
    }

private:
    static constexpr int MOST = 4;
    static constexpr std::chrono::microseconds SPIN{100};
    // wake what sleeps.  A thread counts itself asleep before it looks at turn,
    // calls and stop for the last time, and the caller changes these before it
    // reads the count, so one of the two sees the other.
    void rouse()
    {
        if (!asleep.load()) return;
        { std::lock_guard<std::mutex> l(mu); }
        cv.notify_all();
    }
    void part(int k) const
    {
        const size_t each = (size / (have + 1) + 63) & ~(size_t)63, o = each * k;
        if (o < size) std::memcpy(dst + o, src + o, size - o < each || k == have ? size - o : each);
    }
    void work(int k)
    {
        long seen = 0;
        for (;;) {
            const long called = calls.load();
            const auto until = std::chrono::steady_clock::now() + SPIN;
            while (turn.load(std::memory_order_acquire) == seen && !stop && std::chrono::steady_clock::now() < until)
                std::this_thread::yield();
            if (turn.load(std::memory_order_acquire) != seen) {
                seen++;
                part(k);
                left.fetch_sub(1, std::memory_order_release);
                continue;
            }
            std::unique_lock<std::mutex> l(mu);
            asleep.fetch_add(1);
            cv.wait(l, [&] { return stop || turn.load() != seen || calls.load() != called; });
            asleep.fetch_sub(1);
            if (stop && turn.load() == seen) return;
        }
    }
    std::thread t[MOST];
    int have = 0;
    char *dst = nullptr;
    const char *src = nullptr;
    size_t size = 0;
    std::mutex mu;
    std::condition_variable cv;
    std::atomic<bool> stop{false};
    std::atomic<long> turn{0}, calls{0};
    std::atomic<int> left{0}, asleep{0};
};

}  // namespace st

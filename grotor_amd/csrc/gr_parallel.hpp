// Host loops of the C ABI on several threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace grotor {

// step() on up to `threads` threads, the caller's among them, until it returns
// false; the first exception thrown by any call is rethrown once all have
// stopped.  Where no further thread can be started (a process or memory limit)
// those that run do the work.
template <class Step>
void parallel_steps(int threads, Step&& step) {
    std::atomic<bool> failed{false};
    std::exception_ptr error;
    std::mutex m;
    auto work = [&] {
        try {
            while (!failed.load(std::memory_order_relaxed) && step()) {}
        } catch (...) {
            std::lock_guard<std::mutex> lock(m);
            if (!error) error = std::current_exception();
            failed = true;
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(size_t(std::max(threads, 1)));
    try {
        for (int t = 1; t < threads; ++t) pool.emplace_back(work);
    } catch (const std::system_error&) {
    } catch (const std::bad_alloc&) {
    }
    work();
    for (auto& t : pool) t.join();
    if (error) std::rethrow_exception(error);
}

// f(k) for k in [0, n) on up to 16 host threads (chunks of 256 items).
template <class F>
void parallel_items(int n, F&& f) {
    const int threads = std::max(1, std::min<int>(16, int(std::thread::hardware_concurrency())));
    if (n < 4096 || threads == 1) {
        for (int k = 0; k < n; ++k) f(k);
        return;
    }
    std::atomic<int> next{0};
    parallel_steps(threads, [&] {
        const int k0 = next.fetch_add(256);
        for (int k = k0; k < std::min(n, k0 + 256); ++k) f(k);
        return k0 < n;
    });
}

// f(0) .. f(n - 1) for a few heavy items, one at a time per thread.
template <class F>
void parallel_tasks(int n, F&& f) {
    const int threads = std::max(1, std::min<int>({16, n, int(std::thread::hardware_concurrency())}));
    if (threads <= 1) {
        for (int k = 0; k < n; ++k) f(k);
        return;
    }
    std::atomic<int> next{0};
    parallel_steps(threads, [&] {
        const int k = next++;
        if (k < n) f(k);
        return k < n;
    });
}

}  // namespace grotor

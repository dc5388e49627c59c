// Host loops over several threads.
#pragma once

#include <atomic>
#include <cstddef>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace pbd {

// Runs f(i) for i in [0, n) on up to `threads` threads (each index once).  Where
// the system has no more threads, fewer do the work.  The first exception of any
// of them is thrown here once all have ended; indices not begun by then are left
// out.
template <class F>
void parallel_for(size_t n, unsigned threads, F&& f) {
    std::atomic_size_t next{0};
    std::exception_ptr failed;
    std::mutex failing;
    auto work = [&]() {
        try {
            for (size_t i; (i = next.fetch_add(1)) < n;) f(i);
        } catch (...) {
            next = n;
            std::lock_guard<std::mutex> lock(failing);
            if (!failed) failed = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve(threads);
        for (unsigned t = 1; t < threads && t < n; t++) pool.emplace_back(work);
    } catch (const std::exception&) {
        // no more threads, or no memory for them: those that run do the rest
    }
    work();
    for (auto& th : pool) th.join();
    if (failed) std::rethrow_exception(failed);
}

}  // namespace pbd

// steppe_amd/csrc/host_pool.hpp — a loop over independent host work on a few threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace stp {

// f(i) for i = 0 .. n - 1, handed out in order to min(16, hardware threads, n) threads, the
// caller's among them; fewer where the system grants no more.  After an exception no new i is
// begun, and the one of the smallest i is rethrown here, as a plain loop would throw it.
template <class F>
void for_each_index(std::size_t n, F&& f) {
    const std::size_t hw = std::max(1u, std::thread::hardware_concurrency());
    const std::size_t n_threads = std::min<std::size_t>({16, hw, n});
    std::atomic<std::size_t> next{0};
    std::mutex mutex;
    std::exception_ptr error;
    std::size_t error_at = n;
    auto work = [&] {
        for (std::size_t i = next++; i < n; i = next++) {
            try {
                f(i);
            } catch (...) {
                const std::lock_guard<std::mutex> lock(mutex);
                if (i < error_at) {
                    error_at = i;
                    error = std::current_exception();
                }
                next = n;
            }
        }
    };
    std::vector<std::thread> pool;
    if (n_threads > 1) {
        pool.reserve(n_threads - 1);
        try {
            while (pool.size() < n_threads - 1) pool.emplace_back(work);
        } catch (const std::system_error&) {
            // the threads that did start share the work
        }
    }
    work();
    for (std::thread& t : pool) t.join();
    if (error) std::rethrow_exception(error);
}

}  // namespace stp

// Work shared by a few host threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace spgvbd {

// Runs f(0) .. f(n - 1) on up to `most` host threads, this one among them, and returns when all of them are done. Where
// a call throws, no further index is handed out, every thread is joined, and the first exception is thrown here. Threads
// that cannot be had (their number is limited, or no memory for them) are done without.
template <class F>
void forAll(int64_t n, int most, F &&f)
{
    std::atomic<int64_t> next{0};
    std::exception_ptr error;
    std::mutex guard;
    auto work = [&] {
        try {
            for (int64_t k; (k = next.fetch_add(1)) < n;) f(k);
        } catch (...) {
            next.store(n);
            const std::lock_guard<std::mutex> lock(guard);
            if (!error) error = std::current_exception();
        }
    };
    std::vector<std::thread> threads;
    try {
        threads.reserve(std::max(most, 1));
        while (static_cast<int64_t>(threads.size()) + 1 < std::min<int64_t>(most, n)) threads.emplace_back(work);
    } catch (const std::exception &) {
    }
    work();
    for (auto &t : threads) t.join();
    if (error) std::rethrow_exception(error);
}

}  // namespace spgvbd

// Host loops over up to 16 threads, the caller's own among them.
#pragma once

#include <algorithm>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace pfgpu {

// f(part, parts) for every part.  An exception of a part is thrown here, once
// every part has ended; parts for which no thread is to be had are the caller's.
template <typename F> void parallel_parts(F &&f)
{
    const int parts = int(std::clamp(std::thread::hardware_concurrency(), 1u, 16u));
    std::exception_ptr error;
    std::mutex mutex;
    auto run = [&](int part) {
        try {
            f(part, parts);
        } catch (...) {
            std::lock_guard<std::mutex> lock(mutex);
            if (!error) error = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(size_t(parts));
    int next = 1;
    try {
        for (; next < parts; ++next) pool.emplace_back(run, next);
    } catch (...) {
        // std::system_error or std::bad_alloc: no more threads
    }
    run(0);
    for (; next < parts; ++next) run(next);
    for (std::thread &t : pool) t.join();
    if (error) std::rethrow_exception(error);
}

// f(begin, end) over consecutive runs of 0 .. n-1
template <typename F> void parallel_ranges(int n, F &&f)
{
    parallel_parts([&](int part, int parts) { f(int(int64_t(n) * part / parts), int(int64_t(n) * (part + 1) / parts)); });
}

} // namespace pfgpu

// Host work shared by a few threads. Host code without HIP.
#pragma once

#include <algorithm>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace hoefem {

// f(0) .. f(n - 1), each on its own thread as far as threads can be had. An exception of any of them is thrown
// again here once all have ended (left in a thread it would end the process).
template <class F>
void run_on_threads(int n, F f) {
    std::exception_ptr error;
    std::mutex mu;
    auto part = [&](int i) noexcept {
        try {
            f(i);
        } catch (...) {
            std::lock_guard<std::mutex> lock(mu);
            if (!error) error = std::current_exception();
        }
    };
    std::vector<std::thread> threads;
    int started = 1;
    try {
        for (; started < n; ++started) threads.emplace_back(part, started);
    } catch (...) {  // fewer threads than asked for: their shares here
    }
    part(0);
    for (int i = started; i < n; ++i) part(i);
    for (std::thread& t : threads) t.join();
    if (error) std::rethrow_exception(error);
}

// threads for `work` units, of which `each` are worth one
inline int thread_count(int64_t work, int64_t each) {
    const int64_t most = std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
    return (int)std::max<int64_t>(1, std::min(most, work / each));
}

}  // namespace hoefem

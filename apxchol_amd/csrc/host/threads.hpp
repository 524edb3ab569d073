// Host threads for setup work that runs with fewer of them just as well: where
// the process may not start another, the calling thread does the work.
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace apxchol_amd {

// job(0) .. job(n - 1), side by side where threads can be had; rethrows the
// first exception once all have ended.
template <class F>
void side_by_side(int n, const F& job) {
    std::vector<std::exception_ptr> failed(static_cast<std::size_t>(n));
    std::vector<std::thread> threads;
    threads.reserve(static_cast<std::size_t>(n));
    const auto call = [&](int k) {
        try {
            job(k);
        } catch (...) {
            failed[static_cast<std::size_t>(k)] = std::current_exception();
        }
    };
    int started = 1;   // job 0 and those without a thread are this one's
    try {
        for (; started < n; ++started) threads.emplace_back(call, started);
    } catch (...) {   // no thread, or no memory for one
    }
    call(0);
    for (int k = started; k < n; ++k) call(k);
    for (auto& t : threads) t.join();
    for (const auto& f : failed)
        if (f) std::rethrow_exception(f);
}

}  // namespace apxchol_amd

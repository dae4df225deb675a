// Host work shared among a few threads.
#pragma once

#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace hgdg {

// work(0) .. work(n - 1), each on a thread of its own but work(0), which the
// calling thread does. Where a thread cannot be started (no more of them, or no
// memory for one) the calling thread does its work too. Returns when all have
// ended; the first exception of any goes on from here.
template <typename Work>
void on_threads(int n, Work&& work) {
    std::vector<std::exception_ptr> failed(static_cast<size_t>(n));
    std::vector<std::thread> threads;
    threads.reserve(static_cast<size_t>(n));
    auto guarded = [&](int w) {
        try {
            work(w);
        } catch (...) {
            failed[size_t(w)] = std::current_exception();
        }
    };
    int started = 1;
    try {
        for (; started < n; ++started) threads.emplace_back(guarded, started);
    } catch (...) {  // those that were started run on and are joined below
    }
    guarded(0);
    for (int w = started; w < n; ++w) guarded(w);
    for (std::thread& t : threads) t.join();
    for (const std::exception_ptr& f : failed)
        if (f) std::rethrow_exception(f);
}

}  // namespace hgdg

// Host loops over a few threads.  Plain C++ (host), shared by the library and
// its CPU checks.
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace ssgpu {

// f(share, thread) for every share in [0, shares), taken in turn by at most
// `threads` threads, this one (thread 0) among them.  Threads that cannot be
// started are done without.  An exception ends the loop on every thread and
// leaves here, on the calling thread, once all have ended.
template <typename F> void each_share(int shares, int threads, F&& f) {
    std::atomic<int> next{0};
    std::atomic<bool> stop{false};
    std::exception_ptr err;
    std::mutex mu;
    auto work = [&](int t) noexcept {
        try {
            for (int s = next++; s < shares && !stop; s = next++) f(s, t);
        } catch (...) {
            stop = true;
            std::lock_guard<std::mutex> lk(mu);
            if (!err) err = std::current_exception();
        }
    };
    std::vector<std::thread> th;
    try {
        th.reserve(std::max(0, threads - 1));
        for (int t = 1; t < threads; ++t) th.emplace_back(work, t);
    } catch (...) {
    }
    work(0);
    for (auto& x : th) x.join();
    if (err) std::rethrow_exception(err);
}

}  // namespace ssgpu

// Host threads of the set-up passes.
#pragma once

#include <exception>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace aphip {

// A thread that runs fn, or one that is not joinable where the system gives none.
template <typename Fn>
std::thread try_thread(Fn &&fn) {
    try {
        return std::thread(std::forward<Fn>(fn));
    } catch (const std::exception &) {  // (no thread, or no memory for one)
        return std::thread();
    }
}

// Runs fn() on the calling thread and on up to `most` - 1 further ones, which share the work by a
// counter of fn's own; fewer where the system gives no more threads.  Returns when all have ended,
// and rethrows the first exception of any of them.
template <typename Fn>
void run_workers(int most, Fn &fn) {
    std::mutex mu;
    std::exception_ptr first;
    auto guarded = [&] {
        try {
            fn();
        } catch (...) {
            std::lock_guard<std::mutex> lock(mu);
            if (!first) first = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    if (most > 1) pool.reserve(most - 1);  // (nothing between a thread's start and its join may throw)
    for (int w = 1; w < most; ++w) {
        std::thread t = try_thread(guarded);
        if (!t.joinable()) break;
        pool.push_back(std::move(t));
    }
    guarded();
    for (std::thread &t : pool) t.join();
    if (first) std::rethrow_exception(first);
}

}  // namespace aphip

// Host work dealt to a few threads.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace chysx {

// fn(i) for every i < n, each on one of at most `threads` threads, this one
// among them; an exception of fn is thrown here.  Threads that cannot be
// started (no memory, no more threads) leave their share to the others.
template <class Fn>
void for_each_on_threads(std::size_t n, std::size_t threads, const Fn& fn) {
    threads = std::min<std::size_t>({threads, n, std::max(1u, std::thread::hardware_concurrency())});
    std::atomic<std::size_t> next{0};
    std::exception_ptr failed;
    std::mutex mu;
    const auto work = [&]() noexcept {
        try {
            for (std::size_t i; (i = next.fetch_add(1)) < n;) fn(i);
        } catch (...) {
            std::lock_guard<std::mutex> lk(mu);
            failed = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve(threads);
        while (pool.size() + 1 < threads) pool.emplace_back(work);
    } catch (...) {
        // those that run do the work; they are joined below
    }
    work();
    for (std::thread& t : pool) t.join();
    if (failed) std::rethrow_exception(failed);
}

}  // namespace chysx

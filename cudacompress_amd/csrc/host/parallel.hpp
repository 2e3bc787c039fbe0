// Host loops over the tables of a coder call.
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace cca {

// f(i) for i < n, on one thread for every 75 us of work_us and up to 16, so that starting and joining them
// stays a fraction of what they do.  Where no more threads are to be had those that run do the work; what
// f throws comes out of here, once every thread has ended.
// Start: as std::thread's constructor, for tests.
template <class F, class Start>
void parallel_for(size_t n, double work_us, F f, Start start) {
    const size_t hw = std::max(1u, std::thread::hardware_concurrency());
    const size_t nt = std::min<size_t>({hw, n, (size_t)16, (size_t)(work_us / 75.0) + 1});
    if (nt <= 1) {
        for (size_t i = 0; i < n; i++) f(i);
        return;
    }
    std::atomic<size_t> next{0};
    std::exception_ptr error;
    std::mutex error_mutex;
    auto work = [&]() {
        try {
            for (size_t i = next++; i < n; i = next++) f(i);
        } catch (...) {
            next = n;
            std::lock_guard<std::mutex> lock(error_mutex);
            if (!error) error = std::current_exception();
        }
    };
    std::vector<std::thread> threads;
    threads.reserve(nt - 1);
    for (size_t t = 1; t < nt; t++) {
        try {
            threads.push_back(start(work));
        } catch (const std::system_error&) {
            break;
        }
    }
    work();
    for (std::thread& t : threads) t.join();
    if (error) std::rethrow_exception(error);
}
template <class F>
void parallel_for(size_t n, double work_us, F f) {
    parallel_for(n, work_us, f, [](auto& work) { return std::thread(std::ref(work)); });
}

}  // namespace cca

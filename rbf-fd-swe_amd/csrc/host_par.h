// Host loops over nodes or tiles on a few threads (context set-up).
#pragma once

#include <algorithm>
#include <atomic>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace swe {

// Runs the tasks on host threads of their own (in line where no thread can be
// had); an exception in any (out of memory) is thrown again once all are done.
template <typename F>
void in_parallel(int tasks, F f)
{
    std::atomic<bool> failed{false};
    auto guarded = [&](int k) {
        try {
            f(k);
        } catch (...) {
            failed = true;
        }
    };
    std::vector<std::thread> th(tasks > 1 ? tasks - 1 : 0);
    for (int k = 1; k < tasks; ++k) {
        try {
            th[k - 1] = std::thread(guarded, k);
        } catch (const std::system_error &) {
            guarded(k);
        }
    }
    guarded(0);
    for (std::thread &t : th)
        if (t.joinable())
            t.join();
    if (failed)
        throw std::bad_alloc();
}

// f(first, last) over [0, n) in up to 8 ranges of at least `grain` (a thread
// costs ~50 us).
template <typename F>
void parallel_ranges(int n, int grain, F f)
{
    const int nt =
        std::max(1, std::min({n / std::max(1, grain), 8, (int)std::thread::hardware_concurrency()}));
    in_parallel(nt, [&](int k) { f((int)((long)n * k / nt), (int)((long)n * (k + 1) / nt)); });
}

}  // namespace swe

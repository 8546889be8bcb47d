// host_threads.h -- host threads for the length of one call.
#pragma once

#include <thread>

namespace mt {

// work(0) .. work(n - 1), 1 <= n <= N, each on a thread of its own where one can be had
// and the rest on the calling thread; returns when all have ended.  Throws nothing
// (work must not either): whatever a thread that cannot be started throws -- no more
// threads, or no memory for its state -- only leaves its share to the caller.
template <int N, class F> void on_threads(int n, F &work) noexcept
{
    std::thread th[N];
    int started = 1;
    try {
        for (; started < n; ++started) {
            const int t = started;
            th[t] = std::thread([&work, t] { work(t); });
        }
    } catch (...) {
    }
    work(0);
    for (int t = started; t < n; ++t)
        work(t);
    for (int t = 1; t < started; ++t)
        th[t].join();
}

}  // namespace mt

// A range of array elements cut between host threads.  Host code only.
#pragma once

#include <algorithm>
#include <cstddef>
#include <exception>
#include <thread>

namespace xq {

// f(begin, end) over 0 .. n - 1, cut between threads; what no thread could be started for (no thread or no memory for its
// state left) runs here.  f does not throw.
template <typename F>
void in_ranges(size_t n, F f) {
    constexpr size_t kPerThread = size_t{1} << 18;      // doubles: 2 MB
    const size_t parts = std::min<size_t>({4, n / kPerThread, std::max<size_t>(1, std::thread::hardware_concurrency())});
    if (parts <= 1) { f(size_t{0}, n); return; }
    std::thread threads[3];
    size_t done = n / parts;            // the first part is this thread's
    const size_t own = done;
    for (size_t k = 1; k < parts; k++) {
        const size_t end = n * (k + 1) / parts;
        try {
            threads[k - 1] = std::thread(f, done, end);
        } catch (const std::exception &) {
            break;
        }
        done = end;
    }
    f(size_t{0}, own);
    f(done, n);
    for (std::thread &t : threads)
        if (t.joinable()) t.join();
}

}  // namespace xq

// Cuts arrays between threads (pdynamo3_amd/csrc/xq_ranges.h) where the k-th allocation of a thread's state fails.  Exit
// status 0 if every element was taken once each time.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../../pdynamo3_amd/csrc/xq_ranges.h"

static long long failAt = -1;

void *operator new(std::size_t bytes) {
    if (failAt >= 0 && failAt-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(bytes)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main() {
    for (std::size_t n : {std::size_t{0}, std::size_t{1000}, std::size_t{1} << 19, (std::size_t{1} << 20) + 7})
        for (int k = -1; k < 4; k++) {
            std::vector<int> taken(n, 0);
            failAt = k;
            xq::in_ranges(n, [&taken](std::size_t a, std::size_t b) {
                for (std::size_t i = a; i < b; i++) taken[i]++;
            });
            failAt = -1;
            for (std::size_t i = 0; i < n; i++)
                if (taken[i] != 1) { std::printf("%zu %d: element %zu taken %d times\n", n, k, i, taken[i]); return 1; }
        }
    return 0;
}

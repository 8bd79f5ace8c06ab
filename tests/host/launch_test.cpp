// Host check of the fills' launch extents (eik_launch.h): blocks x threads stays within 32 bits for
// any number of elements a device could hold, a grid-stride loop of that grid reaches every element
// exactly once, and up to the bound every element has a thread of its own.  Prints "ok" or the first
// mismatch.
#include <cstdio>
#include <vector>

#include "eik_launch.h"

int main() {
    // three pending buffers of 331 and 700 sources on 201x201x101 nodes (bricks of 4^3), and the bounds
    const int64_t brick = (int64_t)51 * 51 * 26 * 64;
    const int64_t sizes[] = {0, 1, 255, 256, 257, (int64_t)1 << 30, ((int64_t)1 << 30) + 1, 3 * 331 * brick, 3 * 700 * brick,
                             ((int64_t)1 << 32) - 1, (int64_t)1 << 32, ((int64_t)1 << 32) + 1, (int64_t)1 << 38};
    for (int64_t n : sizes) {
        const uint64_t threads = (uint64_t)eik::fill_blocks(n) * eik::kFillThreads;
        if (threads == 0 || threads >> 32) {
            std::printf("%lld elements: %llu threads\n", (long long)n, (unsigned long long)threads);
            return 1;
        }
        if (n <= eik::kFillBlocksMax * eik::kFillThreads && threads < (uint64_t)n) {
            std::printf("%lld elements share %llu threads\n", (long long)n, (unsigned long long)threads);
            return 1;
        }
        // thread t writes t, t + threads, ...: as many elements in all as there are, the last one n - 1
        uint64_t all = 0;
        if (n > 0) {
            const uint64_t full = (uint64_t)n / threads, rest = (uint64_t)n % threads;
            all = full * (threads - rest) + (full + 1) * rest;
        }
        if (all != (uint64_t)n) {
            std::printf("%lld elements: %llu written\n", (long long)n, (unsigned long long)all);
            return 1;
        }
    }
    std::printf("ok\n");
    return 0;
}

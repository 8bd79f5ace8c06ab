// eik_launch.h -- extents of launches whose work is one element a thread, whatever their number.
// Plain host code with no HIP dependency.
#pragma once
#include <stdint.h>

namespace eik {

// A launch's extent (blocks x threads along x) is a 32-bit number, and the pools of one call go beyond
// it (2^32 pending values are 16 GiB of 288): fills run on a bounded grid and stride over the rest.
constexpr int kFillThreads = 256;
constexpr int64_t kFillBlocksMax = (int64_t)1 << 22;  // 2^30 threads; fewer elements get a thread each
inline unsigned fill_blocks(int64_t n) {
    const int64_t b = (n + kFillThreads - 1) / kFillThreads;
    return (unsigned)(b < 1 ? 1 : (b > kFillBlocksMax ? kFillBlocksMax : b));
}

}  // namespace eik

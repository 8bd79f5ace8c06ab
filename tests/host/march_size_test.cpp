// Host check of the march's buffer sizes (eik_march_size.h): over random instance sets of either mode the
// instances' lists follow one another without overlap and end within the buffer, and the bytes per
// source and per node stay what a solver beside the traveltime and key pools may take.  Prints "ok" or
// the first mismatch.
#include <cstdio>
#include <random>
#include <vector>

#include "eik_march_size.h"

using namespace eik;

static int64_t tiles(int nd, int nx, int ny, int nz) {
    const int e = nd == 2 ? 8 : 4;
    auto t = [&](int n) { return (int64_t)((n + e - 1) / e); };
    return t(nx) * t(ny) * (nd == 3 ? t(nz) : 1);
}

static int64_t total(int mode, int64_t t, int ninst, size_t esz) {
    size_t need[kMarchBufs];
    march_bytes(mode, t * ninst, t, ninst, esz, need);
    int64_t b = 0;
    for (size_t n : need) b += (int64_t)n;
    return b;
}

static int check(const char* what, int64_t got, int64_t most) {
    if (got <= most) return 0;
    std::printf("%s: %lld bytes, more than %lld\n", what, (long long)got, (long long)most);
    return 1;
}

int main() {
    std::mt19937 rng(77);
    for (int trial = 0; trial < 4000; trial++) {
        const int ninst = 1 + (int)(rng() % (trial % 4 == 0 ? 700 : 40));
        for (int mode : {kMarchGroup, kMarchDevice}) {
            const int blocks = mode == kMarchDevice ? round_blocks(ninst) : 0;
            int64_t base = 0;
            for (int in = 0; in < ninst; in++) {
                const int64_t t = 1 + (int64_t)(rng() % (trial % 3 == 0 ? 70000 : 60));
                const unsigned nodes = (unsigned)(64 * t);
                const int64_t words = blocks ? 2 * (int64_t)blocks * seg_cap(nodes, (unsigned)blocks) : 2 * (int64_t)list_cap(nodes);
                if (list_start(base, in, blocks) + words > list_start(base + t, in + 1, blocks)) {
                    std::printf("mode %d instance %d of %d overlaps the next\n", mode, in, ninst);
                    return 1;
                }
                base += t;
            }
            size_t need[kMarchBufs];
            march_bytes(mode, base, base, ninst, 8, need);
            if ((size_t)list_start(base, ninst, blocks) * 4 > need[4]) {
                std::printf("mode %d: lists end beyond their buffer\n", mode);
                return 1;
            }
        }
    }
    size_t none[kMarchBufs];
    march_bytes(kMarchNone, 1000, 1000, 10, 8, none);
    for (size_t n : none)
        if (n) return std::printf("the tile solver has march buffers\n"), 1;
    int bad = 0;
    // a workgroup per source: 26 bytes a node, 8 more for the one slowness grid, and 64 KB a source
    bad += check("61x44 x 400", total(kMarchGroup, tiles(2, 61, 44, 1), 400, 8), 400 * (tiles(2, 61, 44, 1) * 64 * 26 + 65600) + tiles(2, 61, 44, 1) * 64 * 8 + 256);
    bad += check("600x400 x 256", total(kMarchGroup, tiles(2, 600, 400, 1), 256, 8), 256 * (tiles(2, 600, 400, 1) * 64 * 26 + 65600) + tiles(2, 600, 400, 1) * 64 * 8 + 256);
    // device rounds: 48 bytes a node beside the slowness, and the segments' constants over 512 blocks
    bad += check("201x201x101 x 16", total(kMarchDevice, tiles(3, 201, 201, 101), 16, 8),
                 16 * tiles(3, 201, 201, 101) * 64 * 49 + (int64_t)(64 << 20));
    if (!bad) std::printf("ok\n");
    return bad;
}

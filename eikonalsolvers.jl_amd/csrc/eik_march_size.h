// eik_march_size.h -- what the buffers of an ordered march hold, and where an instance's lists start in
// them.  Host code without a HIP dependency; the kernels use the same expressions.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#ifdef __HIPCC__
#define EIK_HD __host__ __device__ __forceinline__
#else
#define EIK_HD inline
#endif

namespace eik {

// kMarchNone: the tile solver; kMarchGroup: one workgroup per instance; kMarchDevice: the whole device
// per round
constexpr int kMarchNone = 0, kMarchGroup = 1, kMarchDevice = 2;

// Entries a list is made for: every node once, and some of the duplicates that a round's wakes can
// add (a list is a small part of the grid, apart from the smallest grids).  A march that needs more
// than its lists hold reports it and is solved by the tile solver instead.
EIK_HD unsigned list_cap(unsigned nodes) { return nodes + nodes / 4u + 8192u; }

// Blocks of a round over all instances: two per CU (256 registers a lane; a call on one stream has them all
// resident).  Milliseconds at 256 / 384 / 512 / 768 / 1024 blocks: 60x75x75 sphere x 24 gradient 17.5 / 16.4 /
// 15.4 / 17.5 / 17.7, 120x150x150 sphere x 32 - / - / 83.8 / 91.8 / 98.8, 201x201x101 x 16 60.3 / 59.4 / 58.4
// (64 an instance from there on).
constexpr int kMaxBlocks = 64;  // per instance: a wave scans their words
constexpr int kRoundBlocks = 512;
inline int round_blocks(int ninst) { return std::max(1, std::min(kMaxBlocks, kRoundBlocks / std::max(1, ninst))); }
constexpr int kRoundRun = 1024;  // nodes a block runs per round; more wait

// a device round's list segment holds an equal part of the list, twice over, and what a block's wakes can add
EIK_HD unsigned seg_cap(unsigned nodes, unsigned blocks) { return 2u * (list_cap(nodes) / blocks) + 4096u; }

// List words of the instances before instance `in`, whose nodes start at 64 * tile_base: two lists of list_cap
// entries each (blocks = 0: a workgroup per instance), or two of `blocks` segments.
EIK_HD int64_t list_start(int64_t tile_base, int64_t in, int blocks) {
    const int64_t caps = tile_base * 80 + in * 8192;  // the list_caps of 64-node bricks
    return blocks == 0 ? 2 * caps : 4 * caps + 2 * 4096 * in * (int64_t)blocks;
}

// Bytes of the march's buffers for ninst instances of ntiles bricks in all and stiles bricks of slowness grids:
// values, slowness, pending values, own words or lowered values, lists, counters and segment words, run lists.
// In FP64 a workgroup per instance takes 26 bytes a node and 64 KB an instance, device rounds 44 and up to
// 2.4 MB; a slowness grid 8 bytes a node of its model.
constexpr int kMarchBufs = 7;
inline void march_bytes(int mode, int64_t ntiles, int64_t stiles, int ninst, size_t esz, size_t* need) {
    const size_t nb = (size_t)ntiles * 64;
    const bool device = mode == kMarchDevice;
    const int blocks = device ? round_blocks(ninst) : 0;
    for (int k = 0; k < kMarchBufs; k++) need[k] = 0;
    if (mode == kMarchNone) return;
    need[0] = nb * esz;
    need[1] = (size_t)stiles * 64 * esz;
    need[2] = (device ? 3 : 1) * nb * sizeof(unsigned);
    need[3] = nb * sizeof(unsigned);
    need[4] = (size_t)list_start(ntiles, ninst, blocks) * sizeof(unsigned);
    need[5] = 256 + (device ? (4 * kMaxBlocks + 2 * (size_t)blocks) * (size_t)ninst * sizeof(unsigned) : 0);
    need[6] = device ? (size_t)ninst * blocks * (kRoundRun + 1) * sizeof(unsigned) : 0;
}

}  // namespace eik

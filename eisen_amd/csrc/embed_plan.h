// Which workgroup of the position index's one launch an id goes to, and the grid of the scatter along the index (embed.hip).
#pragma once
#include <algorithm>
#include <cstddef>

// The index in one launch: kBuckets workgroups, each with one id of every kBuckets in a row (a slot), at most kBucketSlots of them.
constexpr int kBucketBits = 8, kBuckets = 1 << kBucketBits, kBucketSlots = 960;
// Which one moves on by an odd number from slot to slot: ids that are all multiples of a power of two, or of anything else, still spread over the workgroups.
// (With the same one of every slot, the low bits alone, such ids were one workgroup's: 65536 multiples of 256, rows of 64 bf16, index and scatter 812 us, now 47;
// 16384 ids in four residues mod 256, rows of 256, 43 / 19.  It costs 0.3 us of the index of 16384 ids, 7.9 / 8.2.)
constexpr int kBucketStep = 211;
constexpr int scatter_bucket_of(int id) { return ((unsigned)id + ((unsigned)id >> kBucketBits) * kBucketStep) & (kBuckets - 1); }
constexpr int scatter_bucket_id(int slot, int bucket) { return slot << kBucketBits | ((bucket - slot * kBucketStep) & (kBuckets - 1)); }

// The scatter along the index: workgroups of five waves, the first long_blocks for the long runs, one for every long run and 64 columns that there can be, up to four per CU;
// the others a wave per `window` places and 256 columns (small batches: windows of 2 places, the waves are there).
constexpr int kRunThreads = 320, kRunWaves = kRunThreads / 64, kRunWindow = 8;
constexpr size_t kRunBlocksMax = size_t(1) << 23;  // short_blocks of one launch, whose threads are fewer than 2^32; more of them are several launches
struct ScatterRunsGrid {
    size_t long_blocks, short_blocks, window;
};
inline ScatterRunsGrid scatter_runs_grid(size_t n_ids, size_t hidden) {
    const size_t slabs = (hidden + 255) / 256, window = (n_ids + 1) / 2 * slabs <= 4096 ? 2 : kRunWindow, waves = (n_ids + window - 1) / window * slabs;
    return {std::min<size_t>(1024, (n_ids - 1) / 64 * ((hidden + 63) / 64)), (waves + kRunWaves - 1) / kRunWaves, window};
}

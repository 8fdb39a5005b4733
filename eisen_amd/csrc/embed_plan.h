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

// The scatter along the index: workgroups of five waves, the first long_blocks for the long runs, per 64 columns, the others a wave per `window` places and 256 columns
// (small batches: windows of 2 places, the waves are there).  A run is long if it holds long_marks multiples of 64 among its places: two where all of the batch's that can
// be such runs are on the chip at once (two workgroups to a CU), else three, as a wave does runs of that length as well and there are more waves than such workgroups.
// Index and scatter with two / three, us: 1396 Zipf ids x 1024 bf16 13.7 / 15.9, 2000 ids in runs of 130 x 1024 12.5 / 17.9; 32768 ids in runs of 100 x 1024 57 / 37, of 130
// 55 / 40, of 200 45.5 / 44.8, of 400 40.4 / 40.5; 65536 ids of 512 x 512 67 / 51.  With four runs of 200 and 2000 ids take 24, 32768 of 128 x 512 49 (33).
// More workgroups for them keep the others' waves waiting (1024 / 768 / 512: 32768 in runs of 100 x 1024 39 / 38 / 37, of 200 52 / 52 / 45; 65536 of 256 x 1024 73 / 67 / 71).
constexpr int kRunThreads = 320, kRunWaves = kRunThreads / 64, kRunWindow = 8;
constexpr size_t kRunBlocksMax = size_t(1) << 23;  // short_blocks of one launch, whose threads are fewer than 2^32; more of them are several launches
constexpr size_t kLongBlocks = 512;
struct ScatterRunsGrid {
    size_t long_blocks, short_blocks, window;
    int long_marks;
};
inline ScatterRunsGrid scatter_runs_grid(size_t n_ids, size_t hidden) {
    const size_t slabs = (hidden + 255) / 256, window = (n_ids + 1) / 2 * slabs <= 4096 ? 2 : kRunWindow, waves = (n_ids + window - 1) / window * slabs;
    const size_t marks = (n_ids + 63) / 64, long_slabs = (hidden + 63) / 64;
    const int long_marks = marks / 2 * long_slabs <= kLongBlocks ? 2 : 3;
    return {std::min(kLongBlocks, marks / long_marks * long_slabs), (waves + kRunWaves - 1) / kRunWaves, window, long_marks};
}

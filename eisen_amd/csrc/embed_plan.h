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

// Embedding lookup and the deterministic embedding-gradient scatter.
#include <algorithm>
#include <numeric>

#include "device_utils.cuh"
#include "embed_plan.h"
#include "runtime.h"

namespace {

constexpr int kThreads = 256;

// out[i, :] = W[ids[i], :]   (src/graph/ops/transform.rs:296-303): bytes, moved in the widest words that rows and addresses
// are whole numbers of.
template <typename WORD>
__global__ __launch_bounds__(kThreads) void gather_kernel(const WORD* __restrict__ w, const int32_t* __restrict__ ids,
                                                          WORD* __restrict__ out, size_t total, int per_row) {
    for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < total; c += (size_t)gridDim.x * blockDim.x) {
        const size_t i = c / per_row;
        out[c] = w[(size_t)ids[i] * per_row + (int)(c % per_row)];
    }
}
template <typename WORD>
void launch_gather(eisen_ctx* ctx, const void* w, const int32_t* ids, void* out, size_t n_ids, size_t row_bytes) {
    const size_t per_row = row_bytes / sizeof(WORD), total = n_ids * per_row;
    const unsigned blocks = (unsigned)std::min<size_t>(256 * 16, eisen_ceil_div(total, kThreads));
    gather_kernel<WORD><<<blocks, kThreads, 0, ctx->stream>>>((const WORD*)w, ids, (WORD*)out, total, (int)per_row);
}

// One wave owns (one touched vocabulary row) x (one 64-packet column slab) and adds that
// row's occurrences in ascending position order, starting from the value already in gw:
//   gw[row] = ((gw[row] + go[i1]) + go[i2]) + ...      i1 < i2 < ...
// which is the CPU arm's order (src/graph/ops/transform.rs:309-314).  No atomics, so the
// result does not depend on scheduling.  Loads of the next occurrences are issued before the
// adds of the current ones (unroll 4) to keep several rows in flight.
template <typename T>
__global__ __launch_bounds__(kThreads) void scatter_rows_kernel(const T* __restrict__ go, float* __restrict__ gw,
                                                                const int32_t* __restrict__ seg_row,
                                                                const int32_t* __restrict__ seg_begin,
                                                                const int32_t* __restrict__ order, int n_segments,
                                                                int hidden, int slabs) {
    constexpr int N = Pack<T>::N;
    const int lane = threadIdx.x & 63;
    const size_t wave = (size_t)blockIdx.x * (kThreads / kWave) + (threadIdx.x >> 6);
    const size_t seg = wave / slabs;
    if (seg >= (size_t)n_segments) return;
    const int col = ((int)(wave % slabs) * kWave + lane) * N;
    if (col >= hidden) return;
    const size_t row = (size_t)seg_row[seg];
    const int begin = seg_begin[seg], end = seg_begin[seg + 1];
    float acc[N];
    float* dst = gw + row * hidden + col;
#pragma unroll
    for (int j = 0; j < N; j += 4) {
        const float4 v = *reinterpret_cast<const float4*>(dst + j);
        acc[j] = v.x; acc[j + 1] = v.y; acc[j + 2] = v.z; acc[j + 3] = v.w;
    }
    int k = begin;
    for (; k + 4 <= end; k += 4) {
        Pack<T> p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) p[u] = load_pack(go + (size_t)order[k + u] * hidden + col);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int j = 0; j < N; j++) acc[j] += p[u].get(j);
    }
    for (; k < end; k++) {
        const Pack<T> p = load_pack(go + (size_t)order[k] * hidden + col);
#pragma unroll
        for (int j = 0; j < N; j++) acc[j] += p.get(j);
    }
#pragma unroll
    for (int j = 0; j < N; j += 4) *reinterpret_cast<float4*>(dst + j) = make_float4(acc[j], acc[j + 1], acc[j + 2], acc[j + 3]);
}

// Fallback for hidden sizes that are not packet multiples: one thread per (segment, column).
template <typename T>
__global__ __launch_bounds__(kThreads) void scatter_rows_scalar_kernel(const T* __restrict__ go, float* __restrict__ gw,
                                                                       const int32_t* __restrict__ seg_row,
                                                                       const int32_t* __restrict__ seg_begin,
                                                                       const int32_t* __restrict__ order, int n_segments,
                                                                       int hidden) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t seg = t / hidden;
    if (seg >= (size_t)n_segments) return;
    const int col = (int)(t % hidden);
    float acc = gw[(size_t)seg_row[seg] * hidden + col];
    for (int k = seg_begin[seg]; k < seg_begin[seg + 1]; k++) acc += to_f32(go[(size_t)order[k] * hidden + col]);
    gw[(size_t)seg_row[seg] * hidden + col] = acc;
}

// ---- position index built on the device ---------------------------------------------------------
// index = [ids | positions], n ints each: the positions of every id stand together, in ascending order, beside the id (in which order
// the ids follow one another is each builder's own).  Ids outside [0, vocab) stand behind all others as kNoId and belong to no run.
constexpr int kNoId = 0x7fffffff;
constexpr size_t kIndexMax = size_t(1) << 20;  // ids of a batch that is indexed on the device

// One launch: 256 workgroups, each with one id of every 256 in a row (scatter_bucket_of).  All of them read the whole batch (128 KB from the L2s for
// 32768 ids), count what lies before their part and, per id and wave, their own, and place their positions; a wave's ids are consecutive, so the
// places of an id ascend.  What bounds it is the dozen instructions per id and workgroup.  Chunks sorted by a bitonic network, merged and
// listed in three launches had taken 30 us for 32768 ids, 20.4 for 16384, one chunk of up to 1024 and 2048 7.2 and 11.9; this takes 14.6, 8.2, 5.1 and 5.0.
// Built ahead beside a forward pass (Graph::gather) either hides: whole training steps with the index by sort and merge / by this, us (runs of one side differ by
// 1 to 4 %): two layers of 64 in f32, 64 ids 254 / 253, 1024 273 / 271, 2048 286 / 286; two of 256 in bf16, 512 ids 308 / 309, 2048 372 / 371; two of 512, four
// micro-batches of 1024 1704 / 1703; the ~14 M model, 8192 ids 1526 / 1527.
constexpr int kBucketThreads = 1024, kBucketWaves = kBucketThreads / kWave;
constexpr size_t kBucketMax = 65536, kBucketVocab = (size_t)kBuckets * kBucketSlots;
__global__ __launch_bounds__(kBucketThreads) void scatter_bucket_kernel(const int32_t* __restrict__ ids, int n, int vocab, int32_t* __restrict__ out_ids,
                                                                       int32_t* __restrict__ order, int32_t* __restrict__ first_bad) {
    extern __shared__ int places[];  // [wave][slot]: how many the wave has of it, then where its next one goes
    __shared__ int sums[kBucketWaves][2];
    constexpr int LIST = 512;
    __shared__ int list[kBucketWaves][LIST];  // a wave's own ids, slot | index << 10, in order
    static_assert(kBucketWaves * (kBucketSlots + LIST + 2) * sizeof(int) <= 160 << 10, "92 KB for the largest vocabulary, of a CU's 160 KB");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), bucket = blockIdx.x;
    const int here = (vocab + kBuckets - 1) >> kBucketBits;  // slots
    // (an odd number of 256-byte lines: the waves, and with them all workgroups, would otherwise ask one channel of the L2 at a time)
    const int share = ((n + kBucketWaves * kWave - 1) / (kBucketWaves * kWave) | 1) * kWave;
    const int from = wave * share, to = min(n, from + share);
    int* const mine = places + wave * here;
    for (int i = tid; i < kBucketWaves * here; i += kBucketThreads) places[i] = 0;
    __syncthreads();
    constexpr int U = 8;
    int before = 0, bad = kNoId, own = 0;  // before: of smaller buckets, per lane
    for (int i0 = from; i0 < to; i0 += U * kWave) {
        int id[U];
#pragma unroll
        for (int u = 0; u < U; u++) id[u] = ids[min(i0 + u * kWave + lane, n - 1)];
        if (i0 + U * kWave > to)
#pragma unroll
            for (int u = 0; u < U; u++) id[u] = i0 + u * kWave + lane < to ? id[u] : -1;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int b = (unsigned)id[u] < (unsigned)vocab ? scatter_bucket_of(id[u]) : kBuckets;
            before += b < bucket;
            const unsigned long long hits = __ballot(b == bucket);
            if (hits) {
                if (b == bucket) {
                    atomicAdd(&mine[id[u] >> kBucketBits], 1);
                    const int k = own + __popcll(hits & ((1ull << lane) - 1));
                    if (k < LIST) list[wave][k] = id[u] >> kBucketBits | (i0 + u * kWave + lane) << 10;
                }
                own += __popcll(hits);
            }
        }
        if (bucket == 0 && bad == kNoId) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * kWave + lane;
                const unsigned long long wrong = __ballot(i < to && (unsigned)id[u] >= (unsigned)vocab);
                if (wrong) bad = min(bad, i0 + u * kWave + __ffsll(wrong) - 1);
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    if (lane == 0) { sums[wave][0] = before; sums[wave][1] = bucket == 0 ? bad : own; }
    __syncthreads();
    before = 0;
#pragma unroll
    for (int w = 0; w < kBucketWaves; w++) before += sums[w][0];
    if (bucket == 0 && tid == 0 && first_bad) {
        for (int w = 0; w < kBucketWaves; w++) bad = min(bad, sums[w][1]);
        *first_bad = bad;
    }
    if (bucket == kBuckets - 1) {
        int valid = before;
        for (int w = 0; w < kBucketWaves; w++) valid += sums[w][1];
        for (int i = valid + tid; i < n; i += kBucketThreads) {
            out_ids[i] = kNoId;
            order[i] = 0;
        }
    }
    // where the first position of each id goes: thread t takes id t
    int count[kBucketWaves], total = 0;
#pragma unroll
    for (int w = 0; w < kBucketWaves; w++) {
        count[w] = tid < here ? places[w * here + tid] : 0;
        total += count[w];
    }
    int upto = total;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int other = __shfl_up(upto, o, 64);
        if (lane >= o) upto += other;
    }
    __syncthreads();  // the sums above have been read
    if (lane == 63) sums[wave][0] = upto;
    __syncthreads();
    int at = before + upto - total;
#pragma unroll
    for (int w = 0; w < kBucketWaves; w++) at += w < wave ? sums[w][0] : 0;
    if (tid < here) {
#pragma unroll
        for (int w = 0; w < kBucketWaves; w++) {
            places[w * here + tid] = at;
            at += count[w];
        }
    }
    __syncthreads();
    if (own <= LIST) {
        for (int k0 = 0; k0 < own; k0 += kWave) {
            const int these = min(kWave, own - k0), entry = list[wave][min(k0 + lane, own - 1)], slot = entry & 1023;
            int rank = 0, all = 0;  // among the lanes with this id: those before this one, and all
            unsigned long long left = these == kWave ? ~0ull : (1ull << these) - 1;
            while (left) {
                const unsigned long long same = __ballot(slot == __builtin_amdgcn_readlane(slot, __ffsll(left) - 1)) & left;
                if (same >> lane & 1) {
                    rank = __popcll(same & ((1ull << lane) - 1));
                    all = __popcll(same);
                }
                left &= ~same;
            }
            if (lane < these) {
                const int place = mine[slot] + rank;
                out_ids[place] = scatter_bucket_id(slot, bucket);
                order[place] = (int)((unsigned)entry >> 10);
                if (rank == all - 1) mine[slot] = place + 1;  // (a wave's reads of the step above are done)
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        return;
    }
    for (int i0 = from; i0 < to; i0 += U * kWave) {  // hot ids: once more through the batch
        int id[U];
#pragma unroll
        for (int u = 0; u < U; u++) id[u] = ids[min(i0 + u * kWave + lane, n - 1)];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u * kWave + lane;
            unsigned long long left = __ballot(i < to && id[u] >= 0 && id[u] < vocab && scatter_bucket_of(id[u]) == bucket);
            while (left) {  // the lanes with the id of the first one that is left: places in a row
                const int this_id = __builtin_amdgcn_readlane(id[u], __ffsll(left) - 1);
                const unsigned long long same = __ballot(id[u] == this_id) & left;
                const int next = mine[this_id >> kBucketBits];
                if (same >> lane & 1) {
                    const int place = next + __popcll(same & ((1ull << lane) - 1));
                    out_ids[place] = this_id;
                    order[place] = i;
                }
                if (lane == 0) mine[this_id >> kBucketBits] = next + __popcll(same);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                left &= ~same;
            }
        }
    }
}

// Batches and vocabularies beyond that.
// Keys id * 2^shift + position in the chunk are unique, so sorting them is the stable sort of the positions by id.  One
// workgroup of 1024 threads sorts 1024 * R of them (R = 1..16) with a bitonic network whose keys stay in registers: thread t
// holds elements t, t + 1024, ...; a compare-exchange at distance j >= 1024 pairs two registers of one thread, j < 64 two
// lanes of one wave (a shuffle), and only the distances 64..512 go through LDS (18 to 26 of the 55 to 105 steps).  Workgroup c
// takes the ids of chunk c and writes them and their positions in key order; first_bad (may be null) receives per chunk the
// position of its first id outside [0, vocab), or kNoId.  A batch of one chunk is complete with this kernel.
constexpr int kSortThreads = 1024, kSortMax = 16384;
template <int R>
__global__ __launch_bounds__(kSortThreads) void scatter_sort_kernel(const int32_t* __restrict__ ids_all, int n_all, int shift, int vocab,
                                                                   int32_t* __restrict__ sorted_ids, int32_t* __restrict__ order,
                                                                   int32_t* __restrict__ first_bad) {
    constexpr int NP = kSortThreads * R;
    __shared__ unsigned keys[NP];
    __shared__ int bad;
    const int tid = threadIdx.x;
    const int first = blockIdx.x * NP, n = min(NP, n_all - first);
    const int32_t* ids = ids_all + first;
    if (tid == 0) bad = kNoId;
    __syncthreads();
    unsigned key[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int i = r * kSortThreads + tid;
        unsigned v = 0xffffffffu;
        if (i < n) {
            const int id = ids[i];
            if (id >= 0 && id < vocab) v = ((unsigned)id << shift) | (unsigned)i;
            else atomicMin(&bad, first + i);
        }
        key[r] = v;
    }
#pragma unroll
    for (int k = 2; k <= NP; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= kSortThreads) {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int rp = r ^ (j / kSortThreads);
                    if (rp > r) {  // registers r and rp of this thread: element r * 1024 + tid is the lower one
                        const bool asc = (((r * kSortThreads) & k) == 0);  // bit k of the element index lies in the register part (k > j >= 1024)
                        const unsigned lo = min(key[r], key[rp]), hi = max(key[r], key[rp]);
                        key[r] = asc ? lo : hi;
                        key[rp] = asc ? hi : lo;
                    }
                }
            } else {
                if (j >= 64) {
                    __syncthreads();  // the previous exchange's reads are done
#pragma unroll
                    for (int r = 0; r < R; r++) keys[r * kSortThreads + tid] = key[r];
                    __syncthreads();
                }
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int i = r * kSortThreads + tid;
                    const unsigned other = j >= 64 ? keys[r * kSortThreads + (tid ^ j)] : (unsigned)__shfl_xor((int)key[r], j, 64);
                    const bool keep_min = ((i & j) == 0) == ((i & k) == 0);
                    key[r] = keep_min ? min(key[r], other) : max(key[r], other);
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) keys[r * kSortThreads + tid] = key[r];
    if (tid == 0 && first_bad) first_bad[blockIdx.x] = bad;
    __syncthreads();
    const unsigned mask = (1u << shift) - 1;
    for (int i = tid; i < n; i += kSortThreads) {
        const unsigned k = keys[i];
        sorted_ids[first + i] = k == 0xffffffffu ? kNoId : (int32_t)(k >> shift);
        // the padding keys' positions do not matter: they lie in no run
        order[first + i] = k == 0xffffffffu ? 0 : first + (int32_t)(k & mask);
    }
}

// The sorted chunks become one sorted batch.  An element's place is its place in its own chunk plus, for every earlier chunk,
// the ids there that are not larger and, for every later one, those that are smaller: a binary search each.  What bounds it is
// the latency of a search step on ids that another XCD has just written, so the ends of every chunk's 32 groups are searched
// in LDS and only the last steps, which share a group, go to memory; the four waves of a workgroup share the chunks of 64
// elements, four searches at once each (32768 ids in 16 chunks: 31.5 us with every step in memory, 29 with one thread per
// element searching all chunks, now 11).
constexpr int kGroups = 32, kChunksMax = 64;
__global__ __launch_bounds__(kThreads) void scatter_merge_kernel(const int32_t* __restrict__ chunk_ids, const int32_t* __restrict__ chunk_order, int n,
                                                                int chunk, int32_t* __restrict__ sorted_ids, int32_t* __restrict__ order) {
    constexpr int S = 4, WAVES = kThreads / kWave;
    __shared__ int group_last[kChunksMax * kGroups];
    __shared__ int before[WAVES][kWave];
    const int chunks = (n + chunk - 1) / chunk, group = chunk / kGroups, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = blockIdx.x * kWave + lane, from = min(e, n - 1);
    const int id = chunk_ids[from], own = from / chunk;
    for (int i = threadIdx.x; i < chunks * kGroups; i += kThreads) group_last[i] = chunk_ids[min((i + 1) * group, n) - 1];
    __syncthreads();
    int rank = 0;
    for (int c0 = wave * S; c0 < chunks; c0 += WAVES * S) {
        int at[S], len[S], all[S];  // at: ids known to precede this element; the answer lies in [at, at + len]
        const int32_t* base[S];
#pragma unroll
        for (int u = 0; u < S; u++) {
            const int c = min(c0 + u, chunks - 1);
            all[u] = c0 + u < chunks && c != own ? min(chunk, n - c * chunk) : 0;
            base[u] = chunk_ids + (size_t)c * chunk;
            at[u] = 0;  // whole groups whose last id precedes, for now
        }
#pragma unroll
        for (int half = kGroups / 2; half >= 0; half = half > 1 ? half / 2 : half - 1) {
            const int step = max(half, 1);  // 16, 8, 4, 2, 1 and once more 1: from 31 to 32 groups
            int other[S];
#pragma unroll
            for (int u = 0; u < S; u++) other[u] = group_last[min(c0 + u, chunks - 1) * kGroups + min(at[u] + step, kGroups) - 1];
#pragma unroll
            for (int u = 0; u < S; u++) {
                const int end = at[u] + step;
                const bool precedes = c0 + u < own ? other[u] <= id : other[u] < id;
                at[u] = end <= kGroups && end * group <= all[u] && precedes ? end : at[u];
            }
        }
#pragma unroll
        for (int u = 0; u < S; u++) {
            at[u] *= group;
            len[u] = min(all[u] - at[u], group);
        }
        for (int step = group; step > 0; step >>= 1) {
            int other[S];  // a search that has ended loads an id it knows: no branch stands between the loads
#pragma unroll
            for (int u = 0; u < S; u++) other[u] = base[u][max(at[u] + ((len[u] + 1) >> 1) - 1, 0)];
#pragma unroll
            for (int u = 0; u < S; u++) {
                const int half = (len[u] + 1) >> 1;
                const bool precedes = half > 0 && (c0 + u < own ? other[u] <= id : other[u] < id);
                at[u] += precedes ? half : 0;
                len[u] = precedes ? len[u] - half : max(half - 1, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < S; u++) rank += at[u];
    }
    before[wave][lane] = rank;
    __syncthreads();
    if (wave > 0 || e >= n) return;
    rank = e - own * chunk;
#pragma unroll
    for (int w = 0; w < WAVES; w++) rank += before[w][lane];
    sorted_ids[rank] = id;
    order[rank] = chunk_order[e];
}

// ---- the scatter along the index ----------------------------------------------------------------
// gw[row] = ((gw[row] + go[i1]) + go[i2]) + ... with i1 < i2 < ... (the CPU arm's order, src/graph/ops/transform.rs:309-314):
// a run is one chain of dependent adds per column, whatever the schedule.  What bounds it is how many rows of dOut are in
// flight, and for the hot rows of text (thousands of occurrences) the length of the chain:
//  * a long run, one that holds two or three multiples of 64 among its places in the index (ScatterRunsGrid), is a workgroup's per 64
//    columns: four waves fetch its rows, four rows of four columns to a thread and several stages ahead, and leave them in LDS as f32,
//    the rows of a column side by side; the first wave, a lane to a column, adds: a quarter of an LDS read and one add per row.  With
//    the adding wave among those that fetch, rows in bf16 and read by columns, a run of 16384 took 8.2 ns per row; now 5.8, of which 2
//    are the chain of adds.  What a run costs beside that is its start, three waits in a row: the workgroup marks the long runs of the
//    whole index in LDS once, and finds the next one there.  (With a search of the index for every run, 32768 ids of 256, rows of 1024
//    bf16, took 90 us with the index, and 57 with the runs listed in launches of their own; now 40.  The last turn of a run without
//    requests for rows past its end: such batches 1 to 4 % shorter, but the hot runs of text 5 % longer.)
//  * the short runs that begin in 2 or 8 places in a row are a wave's per 256 columns, all their rows in flight: waves with equal
//    work, and no list of runs.  (A wave to a run, its rows 16 at a time: 1396 ids, rows of 448 bf16, lookup and scatter 25.5 us, now 14.4.)
// 32768 Zipf ids, rows of 1024 bf16, lookup and scatter: 114 -> 92 us, of which lookup 15, index 14.5, scatter 38 (the 4649 occurrences of the first id).
// The first workgroups take the long runs, the others the short ones.  first_bad, if given, points at kNoId or nothing is added.
// Four workgroups to a CU (96 registers in bf16).  With three the hot run of text has a little less beside it, everything else waits: 32768
// Zipf ids x 1024 looked up and scattered from memory 90.9 / 92.2 us, but the scatter alone, three / four, of 32768 ids of 256 x 1024 49.7 / 46.8, of
// 65536 of 512 x 1024 77 / 71, of 8192 of 32000 x 4096 66.4 / 63.9, of 200000 of 1000 x 512 234 / 210.
constexpr int kRunStage = 64;
template <typename T> struct Four { typedef T type __attribute__((ext_vector_type(4))); };
template <typename T> struct Two { typedef T type __attribute__((ext_vector_type(2))); };
// four columns from col on of a row of `hidden`; WIDE: rows are whole packets, else they are whole pairs.  Columns past the end repeat
// the last ones: without a branch around a load the compiler knows how many are in flight.
template <bool WIDE, typename T>
__device__ __forceinline__ typename Four<T>::type load_four(const T* row, int col, int hidden) {
    typename Four<T>::type x;
    if (WIDE) {
        x = *reinterpret_cast<const typename Four<T>::type*>(row + min(col, hidden - 4));
    } else {
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
            const typename Two<T>::type y = *reinterpret_cast<const typename Two<T>::type*>(row + min(col + j, hidden - 2));
            x[j] = y[0];
            x[j + 1] = y[1];
        }
    }
    return x;
}
template <bool WIDE>
__device__ __forceinline__ void store_four(float* row, int col, int hidden, const Four<float>::type& x) {
    if (WIDE) {
        if (col < hidden) *reinterpret_cast<Four<float>::type*>(row + col) = x;
    } else {
#pragma unroll
        for (int j = 0; j < 4; j += 2)
            if (col + j < hidden) *reinterpret_cast<float2*>(row + col + j) = make_float2(x[j], x[j + 1]);
    }
}
// The multiples of 64 among the places of the index, 64 to a word, and for each word the number of long runs whose first multiple lies up to its end.
constexpr int kMarkWords = kIndexMax / 64 / 64;
struct RunLds {
    unsigned long long starts[kMarkWords], goes_on[kMarkWords];  // bit l of word i, multiple 64 * i + l: the first of a long run; the next one is of the same run
    int upto[kMarkWords];
};
// Marks them; how many long runs there are.  All threads of the workgroup.
__device__ __forceinline__ int mark_long_runs(const int32_t* __restrict__ ids, int n, int long_marks, RunLds& lds) {
    constexpr int U = 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, words = ((n + 63) / 64 + 63) / 64;
    for (int w0 = wave; w0 < words; w0 += U * kRunWaves) {
        int x[U][4];  // the multiple before, this one, the next, and the last one that a long run from here on holds at least
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < 4; j++) x[u][j] = ids[min(max(((w0 + u * kRunWaves) * 64 + lane + (j < 3 ? j - 1 : long_marks - 1)) * 64, 0), n - 1)];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int w = w0 + u * kRunWaves, k = w * 64 + lane;
            const bool in = (k + 1) * 64 < n && x[u][1] != kNoId, ahead = k > 0 && x[u][0] == x[u][1];
            const bool is_long = in && (k + long_marks - 1) * 64 < n && x[u][3] == x[u][1];
            const unsigned long long starts = __ballot(is_long && !ahead), goes_on = __ballot(in && x[u][2] == x[u][1]);
            if (lane == 0 && w < words) {
                lds.starts[w] = starts;
                lds.goes_on[w] = goes_on;
            }
        }
    }
    __syncthreads();
    if (wave == 0) {
        int before = 0;
        for (int w0 = 0; w0 < words; w0 += kWave) {
            int upto = w0 + lane < words ? __popcll(lds.starts[w0 + lane]) : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int other = __shfl_up(upto, o, 64);
                if (lane >= o) upto += other;
            }
            if (w0 + lane < words) lds.upto[w0 + lane] = before + upto;
            before += __builtin_amdgcn_readlane(upto, 63);
        }
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(lds.upto[words - 1]);
}
// The number-th of them, [begin, end), and its id.  What the marks leave open of begin and end are 64 places each.
__device__ __forceinline__ void find_long_run(const int32_t* __restrict__ ids, int n, int number, const RunLds& lds, int& begin, int& end, int& id) {
    const int lane = threadIdx.x & 63, words = ((n + 63) / 64 + 63) / 64;
    int word = 0;
    for (int w0 = 0; w0 < words; w0 += kWave) {  // the first word up to whose end there are more
        const unsigned long long hit = __ballot(w0 + lane < words && lds.upto[w0 + lane] > number);
        if (hit) {
            word = w0 + __ffsll(hit) - 1;
            break;
        }
    }
    unsigned long long left = lds.starts[word];
    for (int skip = number - (lds.upto[word] - __popcll(left)); skip > 0; skip--) left &= left - 1;
    const int bit = __ffsll(left) - 1;
    unsigned long long stops = ~lds.goes_on[word] & ~((1ull << bit) - 1);
    int at = word;
    while (!stops) stops = ~lds.goes_on[++at];  // (the last multiple goes on nowhere)
    const int first = __builtin_amdgcn_readfirstlane(word * 64 + bit), last = __builtin_amdgcn_readfirstlane(at * 64 + __ffsll(stops) - 1);
    const int before = first * 64 - 63 + lane, after = last * 64 + 1 + lane;
    const int at_first = ids[first * 64], at_before = ids[max(before, 0)], at_after = ids[min(after, n - 1)];  // (one wait for all three)
    id = __builtin_amdgcn_readfirstlane(at_first);
    begin = first * 64 - 63 + __ffsll(__ballot(before >= 0 && at_before == id)) - 1;
    end = last * 64 + 1 + __popcll(__ballot(after < n && at_after == id));
}
// Where four rows of a column stand in a stage: turned so that 16 lanes in a row meet all banks, be they neighbouring columns (the adding
// wave's) or every fourth (those of the waves that fetch).
__device__ __forceinline__ int stage_at(int column, int quad) { return column * kRunStage + 4 * ((quad + (column >> 2) + 4 * (column & 3)) & 15); }
template <typename T, bool WIDE>
__device__ __forceinline__ void scatter_long_run(const T* __restrict__ go, float* __restrict__ gw, const int32_t* __restrict__ order,
                                                 int hidden, int id, int begin, int end, int col0, float* stage) {
    constexpr int D = sizeof(T) == 2 ? 4 : 3;  // stages of rows on their way, per thread
    constexpr int BUF = 64 * kRunStage;
    const int tid = threadIdx.x, lane = tid & 63;
    // whole turns of D stages: with an exit in between the compiler loses count of the loads in flight and waits for all of them
    const int turns = ((end - begin + kRunStage - 1) / kRunStage + D - 1) / D * D;
    if (tid < kWave) {
        float* dst = gw + (size_t)id * hidden + col0 + lane;
        const bool in = col0 + lane < hidden;
        float acc = in ? *dst : 0.f;
        __builtin_amdgcn_s_setprio(3);  // this wave's adds are what the workgroup takes, and the longest run what the launch takes
        for (int s = 0; s < turns; s++) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // stage s is there
            const int rows = end - begin - s * kRunStage;
            if (rows <= 0) continue;
            const float* from = stage + (s & 1) * BUF;
            float4 x[kRunStage / 4];
#pragma unroll
            for (int r = 0; r < kRunStage / 4; r++) x[r] = *reinterpret_cast<const float4*>(from + stage_at(lane, r));
            __builtin_amdgcn_sched_barrier(0);  // all of them on their way before the first add: a read takes as long as 30 adds
            if (rows >= kRunStage) {
#pragma unroll
                for (int r = 0; r < kRunStage / 4; r++) {
                    acc += x[r].x;
                    acc += x[r].y;
                    acc += x[r].z;
                    acc += x[r].w;
                }
            } else {
#pragma unroll
                for (int r = 0; r < kRunStage; r++) {
                    const float sum = acc + (r % 4 == 0 ? x[r / 4].x : r % 4 == 1 ? x[r / 4].y : r % 4 == 2 ? x[r / 4].z : x[r / 4].w);
                    acc = r < rows ? sum : acc;
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (in) *dst = acc;
    } else {
        const int quad = (tid - kWave) / 16, group = tid % 16, col = col0 + 4 * group;
        typename Four<T>::type v[D][4];
        int at[D][4];  // positions, D stages ahead of the rows: the wait for them is then no wait for rows that are needed later
        auto look_up = [&](int s, int (&to)[4]) {
#pragma unroll
            for (int j = 0; j < 4; j++) to[j] = order[min(begin + s * kRunStage + 4 * quad + j, end - 1)];
        };
        auto fetch = [&](const int (&from)[4], typename Four<T>::type (&rows)[4]) {
#pragma unroll
            for (int j = 0; j < 4; j++) rows[j] = load_four<WIDE>(go + (size_t)from[j] * hidden, col, hidden);
        };
#pragma unroll
        for (int d = 0; d < D; d++) look_up(d, at[d]);
#pragma unroll
        for (int d = 0; d < D; d++) {  // (in the loop's order: the compiler's counts of loads in flight hold for both)
            fetch(at[d], v[d]);
            look_up(D + d, at[d]);
        }
        for (int s0 = 0; s0 < turns; s0 += D) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                const int s = s0 + d;
                float* to = stage + (s & 1) * BUF;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *reinterpret_cast<float4*>(to + stage_at(4 * group + j, quad)) = make_float4((float)v[d][0][j], (float)v[d][1][j], (float)v[d][2][j], (float)v[d][3][j]);
                fetch(at[d], v[d]);  // (past the end: its last row again)
                look_up(s + 2 * D, at[d]);
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the adding wave is done with stage s - 1)
            }
        }
    }
    __syncthreads();  // both stages may be written again
}
template <typename T, bool WIDE>
__global__ __launch_bounds__(kRunThreads, 3) void scatter_runs_kernel(const T* __restrict__ go, float* __restrict__ gw, const int32_t* __restrict__ ids,
                                                                  const int32_t* __restrict__ order, const int32_t* __restrict__ first_bad, int n, int hidden,
                                                                  int long_blocks, int long_marks, int window, int first_block) {
    __shared__ __attribute__((aligned(16))) float stage[2 * 64 * kRunStage];
    __shared__ RunLds marks;
    if (first_bad && *first_bad != kNoId) return;
    const int tid = threadIdx.x, lane = tid & 63;
    if ((int)blockIdx.x < long_blocks) {
        const int slabs = (hidden + 63) / 64, items = mark_long_runs(ids, n, long_marks, marks) * slabs;
        for (int item = blockIdx.x; item < items; item += long_blocks) {
            int begin, end, id;
            find_long_run(ids, n, item / slabs, marks, begin, end, id);
            scatter_long_run<T, WIDE>(go, gw, order, hidden, id, begin, end, item % slabs * 64, stage);
        }
        return;
    }
    typedef Four<float>::type F4;
    constexpr int ROWS = sizeof(T) == 2 ? 32 : 16;  // in flight behind the window (more in f32: fewer waves on a SIMD, also for the long runs)
    const int slabs = (hidden + 255) / 256;
    const int item = __builtin_amdgcn_readfirstlane(((int)blockIdx.x - long_blocks + first_block) * kRunWaves + (tid >> 6));
    const int col = (item % slabs * 64 + lane) * 4;
    F4 acc = {};
    int row = -1;  // of the run that is being added up
    auto row_of = [&](int pos, int u) { return load_four<WIDE>(go + (size_t)__builtin_amdgcn_readlane(pos, u) * hidden, col, hidden); };
    int p = item / slabs * window;
    if (p >= n) return;
    const int i = p + lane, far = ((i + 63) & ~63) + 64 * (long_marks - 1);
    const int id = i < n ? ids[i] : kNoId, ahead = i > 0 && i < n ? ids[i - 1] : -1, behind = far < n ? ids[far] : -1;
    int pos = i < n ? order[i] : 0;
    const unsigned long long in_window = (1ull << window) - 1;
    const unsigned long long past = __ballot(id == kNoId), begins = __ballot(id != kNoId && id != ahead), is_long = __ballot(id != kNoId && id != ahead && id == behind);
    if (!(begins & in_window)) return;
    // from the first run that begins in the window on, up to a long one, or to where the last run ends
    const unsigned long long stop = (is_long & in_window) | (begins & ~in_window) | past;
    const int end = stop ? __ffsll(stop) - 1 : kWave;
    {
        const int from = __ffsll(begins) - 1, to = min(end, window);
        typename Four<T>::type x[kRunWindow];
        F4 g[kRunWindow];
#pragma unroll
        for (int u = 0; u < kRunWindow; u++)
            if (u >= from && u < to) {
                x[u] = row_of(pos, u);
                if (begins >> u & 1) g[u] = load_four<WIDE>(gw + (size_t)__builtin_amdgcn_readlane(id, u) * hidden, col, hidden);
            }
        // all of them have arrived: behind the branches the compiler would wait for everything at each use, the stores in between included
#pragma unroll
        for (int u = 0; u < kRunWindow; u++) asm volatile("" : "+v"(x[u]), "+v"(g[u]));
#pragma unroll
        for (int u = 0; u < kRunWindow; u++)
            if (u >= from && u < to) {
                if (begins >> u & 1) {
                    if (row >= 0) store_four<WIDE>(gw + (size_t)row * hidden, col, hidden, acc);
                    acc = g[u];
                    row = __builtin_amdgcn_readlane(id, u);
                }
#pragma unroll
                for (int j = 0; j < 4; j++) acc[j] += (float)x[u][j];
            }
        if (row < 0) return;
    }
    // what is left of the last run, here and in the next 64 places, whose ids and positions are requested before these rows
    for (int done = window, to = end;;) {
        const int next = p + kWave + lane;
        const bool more = to == kWave && next < n;
        const int next_id = more ? ids[next] : kNoId, next_pos = more ? order[next] : 0;
        for (; done < to; done += ROWS) {
            typename Four<T>::type x[ROWS];
#pragma unroll
            for (int u = 0; u < ROWS; u++)
                if (done + u < to) x[u] = row_of(pos, done + u);
#pragma unroll
            for (int u = 0; u < ROWS; u++) asm volatile("" : "+v"(x[u]));
#pragma unroll
            for (int u = 0; u < ROWS; u++)
                if (done + u < to)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[j] += (float)x[u][j];
        }
        if (to < kWave) break;
        p += kWave;
        pos = next_pos;
        done = 0;
        const unsigned long long other = __ballot(next_id != row);
        to = other ? __ffsll(other) - 1 : kWave;
    }
    store_four<WIDE>(gw + (size_t)row * hidden, col, hidden, acc);
}

// How a batch beyond scatter_bucket_kernel's (a vocabulary above 245760, more than 65536 ids) is sorted: chunks of 1024 << k ids, one workgroup each, whose keys (id,
// position in the chunk) fit 32 bits, and a merge.  A batch of up to 2048 ids is one chunk (index of 1500 and 2048 ids 9.2 us, in two chunks 10.8).  Beyond that short
// chunks beat long ones up to where the merge's searches, which grow with their number, outweigh the sort (chunks of 1024 / 2048, us: index of 2049 ids 10.9 / 14.9,
// 4096 11.6 / 15.7, 8192 12.3 / 16.6, 14000 12.9 / 17.3; index and scatter, rows of 64, of 16385 27.4 / 30.0, 24000 33.6 / 33.2, 32768 36.5 / 35.7, 65536 69 / 58).
// Beyond 65536 ids chunks of 16384.
struct ScatterPlan {
    int per_thread, shift;
    size_t chunk, chunks;
};
bool scatter_plan(size_t n_ids, size_t vocab, ScatterPlan* plan) {
    if (n_ids == 0 || n_ids > kIndexMax) return false;
    const int per_thread = n_ids <= 1024 ? 1 : n_ids <= 2048 ? 2 : n_ids <= kSortMax ? 1 : n_ids <= 65536 ? 2 : 16;
    const int shift = per_thread == 1 ? 10 : per_thread == 2 ? 11 : 14;
    // (the vocabularies that are taken do not depend on which of the two shorter chunks the batch gets)
    if ((unsigned long long)vocab << (n_ids <= 1024 ? 10 : std::max(shift, 11)) >= 0xffffffffull) return false;
    const size_t chunk = (size_t)kSortThreads * per_thread;
    *plan = ScatterPlan{per_thread, shift, chunk, eisen_ceil_div(n_ids, chunk)};
    return true;
}
// The batches whose index a caller may build ahead (eisen_hip_gather_index_dev), and whose ids are not checked here.
bool scatter_index_ahead(size_t n_ids, size_t vocab) {
    if (n_ids == 0 || n_ids > (size_t)kSortMax) return false;
    int sh = 10;
    while ((size_t(1) << sh) < n_ids) sh++;
    return (unsigned long long)vocab << sh < 0xffffffffull;
}
bool scatter_rows_ok(const void* go, const float* gw, size_t hidden) {
    return hidden % 2 == 0 && eisen_aligned(go, 8) && eisen_aligned(gw, 8);
}

// Whether the index is one launch of scatter_bucket_kernel; first_bad is one position then, else one per chunk.
bool scatter_by_bucket(size_t n_ids, size_t vocab) { return n_ids <= kBucketMax && vocab <= kBucketVocab; }

// Builds the index (the first 2 * n_ids ints of it).  first_bad, if asked for, points at what the first kernel has written.
int scatter_launch_index(eisen_ctx* ctx, const int32_t* ids_dev, size_t n_ids, size_t vocab, const ScatterPlan& plan, int32_t* index, int32_t** first_bad) {
    int32_t *sorted_ids = index, *order = index + n_ids, *bad = nullptr;
    if (scatter_by_bucket(n_ids, vocab)) {
        if (first_bad) {
            void* ws = nullptr;
            const int rc = eisen_workspace(ctx, sizeof(int32_t), &ws);
            if (rc) return rc;
            *first_bad = (int32_t*)ws;
        }
        const size_t lds = kBucketWaves * eisen_ceil_div(vocab, (size_t)kBuckets) * sizeof(int);
        scatter_bucket_kernel<<<kBuckets, kBucketThreads, lds, ctx->stream>>>(ids_dev, (int)n_ids, (int)vocab, sorted_ids, order, first_bad ? *first_bad : nullptr);
        EISEN_LAUNCH_CHECK(ctx, "scatter_bucket_kernel");
        return 0;
    }
    int32_t *chunk_ids = sorted_ids, *chunk_order = order;
    if (plan.chunks > 1 || first_bad) {
        void* ws = nullptr;
        const int rc = eisen_workspace(ctx, (2 * n_ids + plan.chunks) * sizeof(int32_t), &ws);
        if (rc) return rc;
        bad = (int32_t*)ws + 2 * n_ids;
        if (plan.chunks > 1) {
            chunk_ids = (int32_t*)ws;
            chunk_order = chunk_ids + n_ids;
        }
    }
    if (first_bad) *first_bad = bad;
    const unsigned wgs = (unsigned)plan.chunks;
    if (plan.per_thread == 1)
        scatter_sort_kernel<1><<<wgs, kSortThreads, 0, ctx->stream>>>(ids_dev, (int)n_ids, plan.shift, (int)vocab, chunk_ids, chunk_order, bad);
    else if (plan.per_thread == 2)
        scatter_sort_kernel<2><<<wgs, kSortThreads, 0, ctx->stream>>>(ids_dev, (int)n_ids, plan.shift, (int)vocab, chunk_ids, chunk_order, bad);
    else
        scatter_sort_kernel<16><<<wgs, kSortThreads, 0, ctx->stream>>>(ids_dev, (int)n_ids, plan.shift, (int)vocab, chunk_ids, chunk_order, bad);
    EISEN_LAUNCH_CHECK(ctx, "scatter_sort_kernel");
    return 0;
}
int scatter_launch_merge(eisen_ctx* ctx, size_t n_ids, size_t vocab, const ScatterPlan& plan, int32_t* index) {
    if (plan.chunks == 1 || scatter_by_bucket(n_ids, vocab)) return 0;
    void* ws = nullptr;  // what scatter_launch_index filled: the same block, nothing has asked for a larger one since
    const int rc = eisen_workspace(ctx, (2 * n_ids + plan.chunks) * sizeof(int32_t), &ws);
    if (rc) return rc;
    int32_t *sorted_ids = index, *order = index + n_ids;
    scatter_merge_kernel<<<(unsigned)eisen_ceil_div(n_ids, (size_t)kWave), kThreads, 0, ctx->stream>>>((const int32_t*)ws, (const int32_t*)ws + n_ids, (int)n_ids,
                                                                                                     (int)plan.chunk, sorted_ids, order);
    EISEN_LAUNCH_CHECK(ctx, "scatter_merge_kernel");
    return 0;
}

template <typename T, bool WIDE>
void scatter_launch_runs_as(eisen_ctx* ctx, const int32_t* index, const int32_t* first_bad, const void* go, float* gw, size_t n_ids, size_t hidden) {
    const ScatterRunsGrid g = scatter_runs_grid(n_ids, hidden);
    for (size_t first = 0; first < g.short_blocks; first += kRunBlocksMax) {
        const size_t longs = first == 0 ? g.long_blocks : 0, blocks = longs + std::min(kRunBlocksMax, g.short_blocks - first);
        scatter_runs_kernel<T, WIDE><<<(unsigned)blocks, kRunThreads, 0, ctx->stream>>>((const T*)go, gw, index, index + n_ids, first_bad, (int)n_ids, (int)hidden,
                                                                                       (int)longs, g.long_marks, (int)g.window, (int)first);
    }
}
void scatter_launch_runs(eisen_ctx* ctx, const int32_t* index, const int32_t* first_bad, const void* go, float* gw, int dtype, size_t n_ids, size_t hidden) {
    // whole 16-byte packets of a row where the sizes and addresses give them, pairs of columns otherwise
    const bool wide = hidden % (dtype == EISEN_F32 ? 4 : 8) == 0 && eisen_aligned(go, 16) && eisen_aligned(gw, 16);
    if (dtype == EISEN_F32) {
        if (wide) scatter_launch_runs_as<float, true>(ctx, index, first_bad, go, gw, n_ids, hidden);
        else scatter_launch_runs_as<float, false>(ctx, index, first_bad, go, gw, n_ids, hidden);
    } else {
        if (wide) scatter_launch_runs_as<bf16_t, true>(ctx, index, first_bad, go, gw, n_ids, hidden);
        else scatter_launch_runs_as<bf16_t, false>(ctx, index, first_bad, go, gw, n_ids, hidden);
    }
}

// ids_dev -> index -> scatter.  With `check` the ids are checked first: the positions of the bad ones come back beside what
// follows, the host waits for that copy alone, and *bad tells that nothing was added.  One position: the scatter itself looks at it
// and is launched before the host knows.
int scatter_device_route(eisen_ctx* ctx, const int32_t* ids_dev, const void* go, float* gw, int dtype, size_t n_ids, size_t vocab, size_t hidden,
                         const ScatterPlan& plan, bool check, bool* bad) {
    *bad = false;
    void* dev = nullptr;
    int rc = eisen_hip_malloc(ctx, 2 * n_ids * sizeof(int32_t), &dev);
    if (rc) return rc;
    {
        // algorithmic bytes: every row of dOut read once, every touched row of the f32 gradient read and written once; the
        // touched rows are not known on the host here, so the entry counts dOut and the index only (a lower bound)
        EisenProfScope prof(ctx, dtype == EISEN_BF16 ? "scatter_rows_bf16" : "scatter_rows_f32",
                            (double)n_ids * (double)hidden * eisen_dtype_size(dtype) + 16.0 * (double)n_ids);
        const bool one = scatter_by_bucket(n_ids, vocab);
        int32_t* first_bad = nullptr;
        rc = scatter_launch_index(ctx, ids_dev, n_ids, vocab, plan, (int32_t*)dev, check ? &first_bad : nullptr);
        int32_t found[kIndexMax / 2048];
        int ticket = -1;
        const size_t chunks = one ? 1 : plan.chunks, found_bytes = chunks * sizeof(int32_t);
        if (!rc && check && eisen_hip_dtoh_begin(ctx, first_bad, found_bytes, &ticket)) {
            ticket = -1;  // every staging slot is taken: a plain copy
            rc = eisen_hip_dtoh(ctx, found, first_bad, found_bytes);
        }
        const int rc_merge = rc ? rc : scatter_launch_merge(ctx, n_ids, vocab, plan, (int32_t*)dev);
        if (!rc_merge && one) scatter_launch_runs(ctx, (const int32_t*)dev, first_bad, go, gw, dtype, n_ids, hidden);
        if (ticket >= 0) rc = eisen_hip_dtoh_finish(ctx, ticket, found, found_bytes);
        if (!rc) rc = rc_merge;
        if (!rc && check)
            for (size_t c = 0; c < chunks; c++) *bad = *bad || found[c] != kNoId;
        if (!rc && !*bad && !one) scatter_launch_runs(ctx, (const int32_t*)dev, nullptr, go, gw, dtype, n_ids, hidden);
    }
    hipError_t e = hipGetLastError();
    const int rc_free = eisen_hip_free(ctx, dev);  // stream-ordered: the block is reused only by later work
    if (rc) return rc;
    if (e != hipSuccess) return eisen_set_error(ctx, (int)e, "scatter kernels: %s", hipGetErrorString(e));
    return rc_free;
}

}  // namespace

extern "C" int eisen_hip_gather(eisen_ctx* ctx, const void* weight, const int32_t* ids, void* out, int dtype,
                                size_t n_ids, size_t vocab, size_t hidden) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, weight && ids && out, EISEN_E_ARG, "gather: null pointer");
    EISEN_REQUIRE(ctx, eisen_dtype_ok(dtype), EISEN_E_ARG, "gather: unknown dtype %d", dtype);
    EISEN_REQUIRE(ctx, vocab > 0 && vocab < (size_t(1) << 31) && hidden > 0 && hidden < (size_t(1) << 30), EISEN_E_SHAPE, "gather: vocab/hidden out of range");
    if (n_ids == 0) return 0;
    EisenProfScope prof(ctx, dtype == EISEN_BF16 ? "gather_bf16" : "gather_f32", 2.0 * (double)n_ids * (double)hidden * eisen_dtype_size(dtype) + 4.0 * (double)n_ids);
    const size_t row = hidden * eisen_dtype_size(dtype);
    auto words_of = [&](size_t n) { return row % n == 0 && eisen_aligned(weight, n) && eisen_aligned(out, n); };
    if (words_of(16)) launch_gather<uint4>(ctx, weight, ids, out, n_ids, row);
    else if (words_of(8)) launch_gather<uint2>(ctx, weight, ids, out, n_ids, row);
    else if (words_of(4)) launch_gather<uint32_t>(ctx, weight, ids, out, n_ids, row);
    else launch_gather<uint16_t>(ctx, weight, ids, out, n_ids, row);
    EISEN_LAUNCH_CHECK(ctx, "gather_kernel");
    return 0;
}

extern "C" int eisen_hip_gather_backward(eisen_ctx* ctx, const int32_t* ids_host, const void* go, float* gw, int dtype,
                                         size_t n_ids, size_t vocab, size_t hidden) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, ids_host && go && gw, EISEN_E_ARG, "gather_backward: null pointer");
    EISEN_REQUIRE(ctx, eisen_dtype_ok(dtype), EISEN_E_ARG, "gather_backward: unknown dtype %d", dtype);
    EISEN_REQUIRE(ctx, vocab > 0 && vocab < (size_t(1) << 31) && hidden > 0 && hidden < (size_t(1) << 30) && n_ids < (size_t(1) << 31),
                  EISEN_E_SHAPE, "gather_backward: sizes out of range");
    if (n_ids == 0) return 0;
    for (size_t i = 0; i < n_ids; i++)
        EISEN_REQUIRE(ctx, ids_host[i] >= 0 && (size_t)ids_host[i] < vocab, EISEN_E_ARG,
                      "gather_backward: id %d at position %zu outside [0, %zu)", ids_host[i], i, vocab);
    ScatterPlan plan;
    if (scatter_rows_ok(go, gw, hidden) && scatter_plan(n_ids, vocab, &plan)) {
        // the index is built on the device: the host only hands the ids over
        void* dids = nullptr;
        int rc = eisen_hip_malloc(ctx, n_ids * sizeof(int32_t), &dids);
        if (rc) return rc;
        rc = eisen_hip_htod(ctx, dids, ids_host, n_ids * sizeof(int32_t));
        bool bad = false;
        if (!rc) rc = scatter_device_route(ctx, (const int32_t*)dids, go, gw, dtype, n_ids, vocab, hidden, plan, false, &bad);
        const int rc_free = eisen_hip_free(ctx, dids);
        return rc ? rc : rc_free;
    }
    // larger batches: stable order of positions by token id on the host, ties keep ascending position
    std::vector<int32_t> order(n_ids);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return ids_host[a] < ids_host[b]; });
    std::vector<int32_t> seg_row, seg_begin;
    for (size_t k = 0; k < n_ids; k++)
        if (k == 0 || ids_host[order[k]] != ids_host[order[k - 1]]) {
            seg_row.push_back(ids_host[order[k]]);
            seg_begin.push_back((int32_t)k);
        }
    seg_begin.push_back((int32_t)n_ids);
    const size_t n_seg = seg_row.size();
    // one upload: [order | seg_row | seg_begin]
    const size_t total = n_ids + n_seg + (n_seg + 1);
    std::vector<int32_t> blob(total);
    std::copy(order.begin(), order.end(), blob.begin());
    std::copy(seg_row.begin(), seg_row.end(), blob.begin() + n_ids);
    std::copy(seg_begin.begin(), seg_begin.end(), blob.begin() + n_ids + n_seg);
    void* dev = nullptr;
    int rc = eisen_hip_malloc(ctx, total * sizeof(int32_t), &dev);
    if (rc) return rc;
    rc = eisen_hip_htod(ctx, dev, blob.data(), total * sizeof(int32_t));
    if (rc) {
        (void)eisen_hip_free(ctx, dev);
        return rc;
    }
    const int32_t* d_order = (const int32_t*)dev;
    const int32_t* d_row = d_order + n_ids;
    const int32_t* d_begin = d_row + n_seg;
    const size_t n = dtype == EISEN_F32 ? 4 : 8;
    const bool vec = hidden % n == 0 && eisen_aligned(go, 16) && eisen_aligned(gw, 16);
    // algorithmic bytes: every row of dOut read once, every touched row of the f32 gradient read and written once
    EisenProfScope prof(ctx, dtype == EISEN_BF16 ? "scatter_rows_bf16" : "scatter_rows_f32",
                        (double)n_ids * (double)hidden * eisen_dtype_size(dtype) + 8.0 * (double)n_seg * (double)hidden + 4.0 * (double)total);
    if (vec) {
        const int slabs = (int)eisen_ceil_div(hidden, (size_t)kWave * n);
        const size_t waves = n_seg * slabs;
        const unsigned blocks = (unsigned)eisen_ceil_div(waves, kThreads / kWave);
        if (dtype == EISEN_F32)
            scatter_rows_kernel<float><<<blocks, kThreads, 0, ctx->stream>>>((const float*)go, gw, d_row, d_begin, d_order, (int)n_seg, (int)hidden, slabs);
        else
            scatter_rows_kernel<bf16_t><<<blocks, kThreads, 0, ctx->stream>>>((const bf16_t*)go, gw, d_row, d_begin, d_order, (int)n_seg, (int)hidden, slabs);
        EISEN_LAUNCH_CHECK(ctx, "scatter_rows_kernel");
    } else {
        const unsigned blocks = (unsigned)eisen_ceil_div(n_seg * hidden, kThreads);
        if (dtype == EISEN_F32)
            scatter_rows_scalar_kernel<float><<<blocks, kThreads, 0, ctx->stream>>>((const float*)go, gw, d_row, d_begin, d_order, (int)n_seg, (int)hidden);
        else
            scatter_rows_scalar_kernel<bf16_t><<<blocks, kThreads, 0, ctx->stream>>>((const bf16_t*)go, gw, d_row, d_begin, d_order, (int)n_seg, (int)hidden);
        EISEN_LAUNCH_CHECK(ctx, "scatter_rows_scalar_kernel");
    }
    return eisen_hip_free(ctx, dev);  // stream-ordered: the block is reused only by later work
}

extern "C" int eisen_hip_gather_backward_dev(eisen_ctx* ctx, const int32_t* ids_dev, const void* go, float* gw, int dtype, size_t n_ids,
                                             size_t vocab, size_t hidden) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, ids_dev && go && gw, EISEN_E_ARG, "gather_backward_dev: null pointer");
    EISEN_REQUIRE(ctx, eisen_dtype_ok(dtype), EISEN_E_ARG, "gather_backward_dev: unknown dtype %d", dtype);
    EISEN_REQUIRE(ctx, vocab > 0 && vocab < (size_t(1) << 31) && hidden > 0 && hidden < (size_t(1) << 30) && n_ids < (size_t(1) << 31),
                  EISEN_E_SHAPE, "gather_backward_dev: sizes out of range");
    if (n_ids == 0) return 0;
    ScatterPlan plan;
    int rc = 0;
    if (scatter_rows_ok(go, gw, hidden) && scatter_plan(n_ids, vocab, &plan)) {
        bool bad = false;
        rc = scatter_device_route(ctx, ids_dev, go, gw, dtype, n_ids, vocab, hidden, plan, !scatter_index_ahead(n_ids, vocab), &bad);
        if (rc || !bad) return rc;
    }
    // shapes the device route does not take (and ids it refused, for the message): the ids come back to the host (this
    // synchronises) for the host-built index
    std::vector<int32_t> host(n_ids);
    rc = eisen_hip_dtoh(ctx, host.data(), ids_dev, n_ids * sizeof(int32_t));
    if (rc) return rc;
    return eisen_hip_gather_backward(ctx, host.data(), go, gw, dtype, n_ids, vocab, hidden);
}

// The two halves of eisen_hip_gather_backward_dev for a caller that knows the ids long before the gradient exists (the token ids
// of a training step are known when its forward pass starts): the index depends on the ids alone.
extern "C" int eisen_hip_gather_index_dev(eisen_ctx* ctx, const int32_t* ids_dev, size_t n_ids, size_t vocab, int32_t* index) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, ids_dev && index, EISEN_E_ARG, "gather_index_dev: null pointer");
    EISEN_REQUIRE(ctx, vocab > 0 && vocab < (size_t(1) << 31), EISEN_E_SHAPE, "gather_index_dev: vocab out of range");
    if (n_ids == 0) return 0;
    ScatterPlan plan;
    EISEN_REQUIRE(ctx, scatter_index_ahead(n_ids, vocab) && scatter_plan(n_ids, vocab, &plan), EISEN_E_SHAPE,
                  "gather_index_dev: %zu ids of a vocabulary of %zu are more than the device-side index takes", n_ids, vocab);
    EisenProfScope prof(ctx, "scatter_index", 16.0 * (double)n_ids);
    const int rc = scatter_launch_index(ctx, ids_dev, n_ids, vocab, plan, index, nullptr);
    return rc ? rc : scatter_launch_merge(ctx, n_ids, vocab, plan, index);
}

extern "C" int eisen_hip_gather_backward_indexed(eisen_ctx* ctx, const int32_t* index, const void* go, float* gw, int dtype, size_t n_ids,
                                                 size_t vocab, size_t hidden) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, index && go && gw, EISEN_E_ARG, "gather_backward_indexed: null pointer");
    EISEN_REQUIRE(ctx, eisen_dtype_ok(dtype), EISEN_E_ARG, "gather_backward_indexed: unknown dtype %d", dtype);
    EISEN_REQUIRE(ctx, vocab > 0 && vocab < (size_t(1) << 31) && hidden > 0 && hidden < (size_t(1) << 30), EISEN_E_SHAPE,
                  "gather_backward_indexed: vocab/hidden out of range");
    if (n_ids == 0) return 0;
    EISEN_REQUIRE(ctx, scatter_rows_ok(go, gw, hidden) && scatter_index_ahead(n_ids, vocab), EISEN_E_SHAPE,
                  "gather_backward_indexed: rows of %zu values at these addresses need eisen_hip_gather_backward_dev", hidden);
    EisenProfScope prof(ctx, dtype == EISEN_BF16 ? "scatter_rows_bf16" : "scatter_rows_f32", (double)n_ids * (double)hidden * eisen_dtype_size(dtype) + 16.0 * (double)n_ids);
    scatter_launch_runs(ctx, index, nullptr, go, gw, dtype, n_ids, hidden);
    EISEN_LAUNCH_CHECK(ctx, "scatter_runs_kernel");
    return 0;
}

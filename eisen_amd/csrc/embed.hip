// Embedding lookup and the deterministic embedding-gradient scatter.
#include <algorithm>
#include <numeric>

#include "device_utils.cuh"
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
// index = [sorted ids | positions in sorted order | runs], n ints each.  The third part lists where the runs of equal ids
// begin, in order, so that run r is [runs[r], runs[r + 1]); after the last run it is filled with the number of valid ids, and
// from its end backwards it holds the number of long runs and their numbers, complemented: ~count, ~r0, ~r1, ...  (A run
// of kLongRun occurrences frees kLongRun - 1 entries, so the two lists never meet; with n runs there is neither filling nor a
// long run.)  Ids outside [0, vocab) sort behind all others as kNoId and belong to no run.
constexpr int kNoId = 0x7fffffff;
constexpr int kLongRun = 128;

// Keys id * 2^shift + position in the chunk are unique, so sorting them is the stable sort of the positions by id.  One
// workgroup of 1024 threads sorts 1024 * R of them (R = 1..16) with a bitonic network whose keys stay in registers: thread t
// holds elements t, t + 1024, ...; a compare-exchange at distance j >= 1024 pairs two registers of one thread, j < 64 two
// lanes of one wave (a shuffle), and only the distances 64..512 go through LDS (18 to 26 of the 55 to 105 steps).  Workgroup c
// takes the ids of chunk c and writes them and their positions in key order; first_bad (may be null) receives per chunk the
// position of its first id outside [0, vocab), or kNoId.  A batch of one chunk is complete with this kernel: it also lists the runs.
constexpr int kSortThreads = 1024, kSortMax = 16384;
template <int R>
__global__ __launch_bounds__(kSortThreads) void scatter_sort_kernel(const int32_t* __restrict__ ids_all, int n_all, int shift, int vocab,
                                                                   int32_t* __restrict__ sorted_ids, int32_t* __restrict__ order,
                                                                   int32_t* __restrict__ runs, int32_t* __restrict__ first_bad) {
    constexpr int NP = kSortThreads * R;
    __shared__ unsigned keys[NP];
    __shared__ int totals[kSortThreads / kWave][2];
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
    if (!runs) return;
    // one chunk: thread t lists the runs that begin in elements [t R, t R + R)
    int begins = 0, longs = 0;
    unsigned begin_bits = 0, long_bits = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int i = tid * R + r;
        if (i >= n || keys[i] == 0xffffffffu) continue;
        const unsigned id = keys[i] >> shift;
        if (i > 0 && (keys[i - 1] >> shift) == id) continue;
        begins++;
        begin_bits |= 1u << r;
        const int last = i + kLongRun - 1;
        if (last < n && keys[last] != 0xffffffffu && (keys[last] >> shift) == id) {
            longs++;
            long_bits |= 1u << r;
        }
    }
    const int lane = tid & 63, wid = tid >> 6;
    int b = begins, l = longs;  // inclusive sums over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int bo = __shfl_up(b, o, 64), lo = __shfl_up(l, o, 64);
        if (lane >= o) { b += bo; l += lo; }
    }
    if (lane == 63) { totals[wid][0] = b; totals[wid][1] = l; }
    __syncthreads();
    int b_all = 0, l_all = 0, b_before = 0, l_before = 0;
#pragma unroll
    for (int w = 0; w < kSortThreads / kWave; w++) {
        if (w == wid) { b_before = b_all; l_before = l_all; }
        b_all += totals[w][0];
        l_all += totals[w][1];
    }
    int at_b = b_before + b - begins, at_l = l_before + l - longs;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (long_bits >> r & 1) runs[n - 2 - at_l++] = ~at_b;
        if (begin_bits >> r & 1) runs[at_b++] = tid * R + r;
    }
    // the number of valid ids: where the padding keys begin
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (keys[mid] != 0xffffffffu) lo = mid + 1;
        else hi = mid;
    }
    for (int i = b_all + tid; i < n - (l_all ? l_all + 1 : 0); i += kSortThreads) runs[i] = lo;
    if (tid == 0 && l_all) runs[n - 1] = ~l_all;
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

// Lists the runs of a merged batch.  A workgroup takes 1024 sorted ids and counts by itself what begins before them (each of
// its threads looks at every 1024th id): a handful of reads per thread instead of a scan over workgroups.
__global__ __launch_bounds__(kSortThreads) void scatter_runs_list_kernel(const int32_t* __restrict__ sorted_ids, int n, int32_t* __restrict__ runs) {
    __shared__ int before[kSortThreads / kWave][3], own[kSortThreads / kWave][2];  // per wave: what it counted before this workgroup's ids, and among them
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int first = blockIdx.x * kSortThreads;
    int b = 0, l = 0, valid = 0;
    for (int i0 = 0; i0 < first; i0 += 8 * kSortThreads) {  // 24 loads in flight: the loop is a chain of load latencies
        int id[8], prev[8], far[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = min(i0 + u * kSortThreads + tid, n - 1);
            id[u] = sorted_ids[i];
            prev[u] = sorted_ids[max(i - 1, 0)];
            far[u] = sorted_ids[min(i + kLongRun - 1, n - 1)];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = i0 + u * kSortThreads + tid;
            if (i >= first || id[u] == kNoId) continue;
            valid++;
            if (i > 0 && prev[u] == id[u]) continue;
            b++;
            l += i + kLongRun <= n && far[u] == id[u];
        }
    }
    const int i = first + tid, own_id = i < n ? sorted_ids[i] : kNoId;
    const bool begins = own_id != kNoId && (i == 0 || sorted_ids[i - 1] != own_id);
    const bool is_long = begins && i + kLongRun <= n && sorted_ids[i + kLongRun - 1] == own_id;
    valid += own_id != kNoId;
    const unsigned long long bm = __ballot(begins), lm = __ballot(is_long), below = (1ull << lane) - 1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        b += __shfl_xor(b, o, 64);
        l += __shfl_xor(l, o, 64);
        valid += __shfl_xor(valid, o, 64);
    }
    if (lane == 0) {
        before[wid][0] = b; before[wid][1] = l; before[wid][2] = valid;
        own[wid][0] = __popcll(bm); own[wid][1] = __popcll(lm);
    }
    __syncthreads();
    int b_at = 0, l_at = 0, b_all = 0, l_all = 0, v_all = 0;
#pragma unroll
    for (int w = 0; w < kSortThreads / kWave; w++) {
        b_at += before[w][0] + (w < wid ? own[w][0] : 0);
        l_at += before[w][1] + (w < wid ? own[w][1] : 0);
        b_all += before[w][0] + own[w][0];
        l_all += before[w][1] + own[w][1];
        v_all += before[w][2];
    }
    b_at += __popcll(bm & below);
    l_at += __popcll(lm & below);
    if (begins) runs[b_at] = i;
    if (is_long) runs[n - 2 - l_at] = ~b_at;
    if (blockIdx.x == gridDim.x - 1) {  // the last workgroup has counted everything
        for (int k = b_all + tid; k < n - (l_all ? l_all + 1 : 0); k += kSortThreads) runs[k] = v_all;
        if (tid == 0 && l_all) runs[n - 1] = ~l_all;
    }
}

// ---- the scatter along the index ----------------------------------------------------------------
// gw[row] = ((gw[row] + go[i1]) + go[i2]) + ... with i1 < i2 < ... (the CPU arm's order, src/graph/ops/transform.rs:309-314):
// a run is one chain of dependent adds per column, whatever the schedule.  What bounds it is how many rows of dOut are in
// flight, and for the hot rows of text (thousands of occurrences) the length of the chain:
//  * a long run (>= kLongRun) is a workgroup's per 64 columns: all four waves fetch the next 32 KB of its rows into registers
//    while one wave adds the rows that stand in LDS;
//  * a short run is a wave's per 64 * C columns, up to 16 rows in flight.
// The first workgroups take the long runs, the others the short ones.
// lane l's column of 32 rows of 64 values in LDS.  bf16: the transposing read hands every lane four rows of its column at once
// (one 2-byte read per row and lane made the adds of a long run cost 24 cycles each).
__device__ __forceinline__ void read_columns(const float* rows, float* x) {
#pragma unroll
    for (int u = 0; u < 32; u++) x[u] = rows[u * 64 + (threadIdx.x & 63)];
}
__device__ __forceinline__ void read_columns(const bf16_t* rows, float* x) {
    typedef bf16x4 __attribute__((address_space(3))) * lds_ptr;
    const int lane = threadIdx.x & 63, L = lane & 15;
    const bf16_t* p = rows + (L >> 2) * 64 + (lane & 48) + 4 * (L & 3);
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const bf16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)(p + u * 256));
#pragma unroll
        for (int j = 0; j < 4; j++) x[4 * u + j] = (float)v[j];
    }
}
template <typename T, int N> struct Cols { typedef T type __attribute__((ext_vector_type(N))); };
template <typename T, bool WIDE>
__global__ __launch_bounds__(kThreads) void scatter_runs_kernel(const T* __restrict__ go, float* __restrict__ gw, const int32_t* __restrict__ sorted_ids,
                                                               const int32_t* __restrict__ order, const int32_t* __restrict__ runs, int n, int hidden) {
    constexpr int E = WIDE ? 16 / (int)sizeof(T) : 2;  // columns per load of a long run
    constexpr int LPR = 64 / E;                        // lanes per row of 64 columns
    constexpr int RPI = kThreads / LPR;                // rows per load of the workgroup
    constexpr int U = sizeof(T) * E == 16 ? 8 : 16;    // loads in flight per thread
    constexpr int ST = RPI * U;                        // rows per stage
    typedef typename Cols<T, E>::type VE;
    __shared__ __attribute__((aligned(16))) T stage[ST * 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int n_long = runs[n - 1] < 0 ? ~runs[n - 1] : 0;
    const int long_slabs = (hidden + 63) / 64;
    const long long long_items = (long long)n_long * long_slabs;
    const int long_blocks = (int)min(long_items, (long long)(gridDim.x / 2));
    if ((int)blockIdx.x < long_blocks) {
        for (long long item = blockIdx.x; item < long_items; item += long_blocks) {
            const int r = ~runs[n - 2 - (int)(item / long_slabs)];
            const int begin = runs[r], end = r + 1 < n ? runs[r + 1] : n;
            const int col0 = (int)(item % long_slabs) * 64;
            const int col = col0 + (tid % LPR) * E, sub = tid / LPR;
            const bool in = col < hidden;  // hidden is a multiple of E
            const T* src = go + (in ? col : 0);
            float* dst = gw + (size_t)sorted_ids[begin] * hidden + col0 + lane;
            float acc = tid < 64 && col0 + lane < hidden ? *dst : 0.f;
            VE v[U];
            int at[U];  // positions of the rows to be fetched next, a stage ahead of the rows
            auto look_up = [&](int k0) {
#pragma unroll
                for (int u = 0; u < U; u++) at[u] = order[min(k0 + u * RPI + sub, end - 1)];
            };
            auto fetch = [&] {
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = *reinterpret_cast<const VE*>(src + (size_t)at[u] * hidden);
            };
            look_up(begin);
            fetch();
            look_up(begin + ST);
            for (int k0 = begin; k0 < end; k0 += ST) {
                __syncthreads();  // the previous stage has been added up
#pragma unroll
                for (int u = 0; u < U; u++) *reinterpret_cast<VE*>(&stage[(u * RPI + sub) * 64 + (tid % LPR) * E]) = v[u];
                __syncthreads();
                if (k0 + ST < end) {
                    fetch();
                    look_up(k0 + 2 * ST);
                }
                if (tid < 64) {
                    const int rows = min(ST, end - k0);
                    int k = 0;
                    for (; k + 32 <= rows; k += 32) {
                        float x[32];
                        read_columns(&stage[k * 64], x);
#pragma unroll
                        for (int u = 0; u < 32; u++) acc += x[u];
                    }
                    for (; k < rows; k++) acc += to_f32(stage[k * 64 + lane]);
                }
            }
            if (tid < 64 && col0 + lane < hidden) *dst = acc;
        }
        return;
    }
    constexpr int C = WIDE ? 4 : 2, F = 16;  // columns per lane, rows in flight
    typedef typename Cols<T, C>::type VC;
    typedef typename Cols<float, C>::type VF;
    const int slabs = (hidden + 64 * C - 1) / (64 * C);
    const int waves = (int)(gridDim.x - long_blocks) * (kThreads / kWave);
    const int item = __builtin_amdgcn_readfirstlane((blockIdx.x - long_blocks) * (kThreads / kWave) + (tid >> 6));
    int r = item / slabs, slab = item % slabs;
    for (; r < n; r += waves / slabs + (slab + waves % slabs >= slabs), slab = (slab + waves % slabs) % slabs) {
        const int begin = runs[r];
        if (begin < 0 || begin >= n) return;
        const int end = r + 1 < n ? runs[r + 1] : n, row = sorted_ids[begin];
        if (end <= begin || row == kNoId) return;  // behind the last run
        if (end - begin >= kLongRun) continue;
        const int col = (slab * 64 + lane) * C;
        if (col >= hidden) continue;  // hidden is a multiple of C
        VF acc = *reinterpret_cast<const VF*>(gw + (size_t)row * hidden + col);
        const T* src = go + col;
        for (int k = begin; k < end; k += F) {
            VC p[F];
#pragma unroll
            for (int u = 0; u < F; u++)
                if (k + u < end) p[u] = *reinterpret_cast<const VC*>(src + (size_t)order[k + u] * hidden);
#pragma unroll
            for (int u = 0; u < F; u++)
                if (k + u < end)
#pragma unroll
                    for (int j = 0; j < C; j++) acc[j] += (float)p[u][j];
        }
        *reinterpret_cast<VF*>(gw + (size_t)row * hidden + col) = acc;
    }
}

// How a batch is sorted: chunks of 1024 << k ids, one workgroup each, whose keys (id, position in the chunk) fit 32 bits.  A
// batch of up to 2048 ids is one chunk, complete with one launch (2048 ids: 11.8 us for the index, 15.6 in two chunks).  Beyond that
// short chunks and a merge beat one long bitonic network, the shorter ones up to where the merge's searches, which grow with the
// number of chunks, outweigh the sort (chunks of 1024 / 2048 / 4096 / all in one, us for the index): 2049 ids 15.7 / 19.7 / 19.5,
// 4096 16.6 / 20.8 / 20.2, 8192 17.7 / 21.9 / 29.8 / 39.6, 16384 20.3 / 24.4 / 32.6 / 85; with the scatter, 24000 ids 62.6 / 62.0, 32768 74.4 / 73.3,
// 65536 141 / 130.  Beyond 65536 ids chunks of 16384.  32768 Zipf ids, rows of 1024 bf16, lookup and scatter: 114 us, of which sort 10,
// merge 11, list of runs 10, scatter 48; with the host's stable_sort and four rows of a run in flight 2790 us.
struct ScatterPlan {
    int per_thread, shift;
    size_t chunk, chunks;
};
constexpr size_t kIndexMax = size_t(1) << 20;
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

// Builds the index (3 * n_ids ints).  first_bad, if asked for, points at plan.chunks ints that the first kernel has written.
int scatter_launch_index(eisen_ctx* ctx, const int32_t* ids_dev, size_t n_ids, size_t vocab, const ScatterPlan& plan, int32_t* index, int32_t** first_bad) {
    int32_t *sorted_ids = index, *order = index + n_ids, *runs = index + 2 * n_ids, *bad = nullptr;
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
    int32_t* runs_now = plan.chunks == 1 ? runs : nullptr;
    const unsigned wgs = (unsigned)plan.chunks;
    if (plan.per_thread == 1)
        scatter_sort_kernel<1><<<wgs, kSortThreads, 0, ctx->stream>>>(ids_dev, (int)n_ids, plan.shift, (int)vocab, chunk_ids, chunk_order, runs_now, bad);
    else if (plan.per_thread == 2)
        scatter_sort_kernel<2><<<wgs, kSortThreads, 0, ctx->stream>>>(ids_dev, (int)n_ids, plan.shift, (int)vocab, chunk_ids, chunk_order, runs_now, bad);
    else
        scatter_sort_kernel<16><<<wgs, kSortThreads, 0, ctx->stream>>>(ids_dev, (int)n_ids, plan.shift, (int)vocab, chunk_ids, chunk_order, runs_now, bad);
    EISEN_LAUNCH_CHECK(ctx, "scatter_sort_kernel");
    return 0;
}
int scatter_launch_merge(eisen_ctx* ctx, size_t n_ids, const ScatterPlan& plan, int32_t* index) {
    if (plan.chunks == 1) return 0;
    void* ws = nullptr;  // what scatter_launch_index filled: the same block, nothing has asked for a larger one since
    const int rc = eisen_workspace(ctx, (2 * n_ids + plan.chunks) * sizeof(int32_t), &ws);
    if (rc) return rc;
    int32_t *sorted_ids = index, *order = index + n_ids, *runs = index + 2 * n_ids;
    scatter_merge_kernel<<<(unsigned)eisen_ceil_div(n_ids, (size_t)kWave), kThreads, 0, ctx->stream>>>((const int32_t*)ws, (const int32_t*)ws + n_ids, (int)n_ids,
                                                                                                     (int)plan.chunk, sorted_ids, order);
    scatter_runs_list_kernel<<<(unsigned)eisen_ceil_div(n_ids, (size_t)kSortThreads), kSortThreads, 0, ctx->stream>>>(sorted_ids, (int)n_ids, runs);
    EISEN_LAUNCH_CHECK(ctx, "scatter_merge_kernel");
    return 0;
}

template <typename T, bool WIDE>
void scatter_launch_runs_as(eisen_ctx* ctx, const int32_t* index, const void* go, float* gw, size_t n_ids, size_t hidden) {
    const size_t slabs = eisen_ceil_div(hidden, (size_t)kWave * (WIDE ? 4 : 2));
    // at most 8 workgroups per CU for the short runs (they stride over the list), and what the long runs can use
    const size_t blocks = std::max<size_t>(2, std::min<size_t>(256 * 8, eisen_ceil_div(n_ids * slabs, (size_t)(kThreads / kWave))) +
                                                  std::min<size_t>(256 * 4, n_ids / kLongRun * eisen_ceil_div(hidden, (size_t)kWave)));
    scatter_runs_kernel<T, WIDE><<<(unsigned)blocks, kThreads, 0, ctx->stream>>>((const T*)go, gw, index, index + n_ids, index + 2 * n_ids, (int)n_ids, (int)hidden);
}
void scatter_launch_runs(eisen_ctx* ctx, const int32_t* index, const void* go, float* gw, int dtype, size_t n_ids, size_t hidden) {
    // whole 16-byte packets of a row where the sizes and addresses give them, pairs of columns otherwise
    const bool wide = hidden % (dtype == EISEN_F32 ? 4 : 8) == 0 && eisen_aligned(go, 16) && eisen_aligned(gw, 16);
    if (dtype == EISEN_F32) {
        if (wide) scatter_launch_runs_as<float, true>(ctx, index, go, gw, n_ids, hidden);
        else scatter_launch_runs_as<float, false>(ctx, index, go, gw, n_ids, hidden);
    } else {
        if (wide) scatter_launch_runs_as<bf16_t, true>(ctx, index, go, gw, n_ids, hidden);
        else scatter_launch_runs_as<bf16_t, false>(ctx, index, go, gw, n_ids, hidden);
    }
}

// ids_dev -> index -> scatter.  With `check` the ids are checked first: the positions of the bad ones come back beside the
// merge, the host waits for that copy alone, and *bad tells that nothing was added.
int scatter_device_route(eisen_ctx* ctx, const int32_t* ids_dev, const void* go, float* gw, int dtype, size_t n_ids, size_t vocab, size_t hidden,
                         const ScatterPlan& plan, bool check, bool* bad) {
    *bad = false;
    void* dev = nullptr;
    int rc = eisen_hip_malloc(ctx, 3 * n_ids * sizeof(int32_t), &dev);
    if (rc) return rc;
    {
        // algorithmic bytes: every row of dOut read once, every touched row of the f32 gradient read and written once; the
        // touched rows are not known on the host here, so the entry counts dOut and the index only (a lower bound)
        EisenProfScope prof(ctx, dtype == EISEN_BF16 ? "scatter_rows_bf16" : "scatter_rows_f32",
                            (double)n_ids * (double)hidden * eisen_dtype_size(dtype) + 16.0 * (double)n_ids);
        int32_t* first_bad = nullptr;
        rc = scatter_launch_index(ctx, ids_dev, n_ids, vocab, plan, (int32_t*)dev, check ? &first_bad : nullptr);
        int32_t found[kIndexMax / 2048];
        int ticket = -1;
        const size_t found_bytes = plan.chunks * sizeof(int32_t);
        if (!rc && check && eisen_hip_dtoh_begin(ctx, first_bad, found_bytes, &ticket)) {
            ticket = -1;  // every staging slot is taken: a plain copy
            rc = eisen_hip_dtoh(ctx, found, first_bad, found_bytes);
        }
        const int rc_merge = rc ? rc : scatter_launch_merge(ctx, n_ids, plan, (int32_t*)dev);
        if (ticket >= 0) rc = eisen_hip_dtoh_finish(ctx, ticket, found, found_bytes);
        if (!rc) rc = rc_merge;
        if (!rc && check)
            for (size_t c = 0; c < plan.chunks; c++) *bad = *bad || found[c] != kNoId;
        if (!rc && !*bad) scatter_launch_runs(ctx, (const int32_t*)dev, go, gw, dtype, n_ids, hidden);
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
    return rc ? rc : scatter_launch_merge(ctx, n_ids, plan, index);
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
    scatter_launch_runs(ctx, index, go, gw, dtype, n_ids, hidden);
    EISEN_LAUNCH_CHECK(ctx, "scatter_runs_kernel");
    return 0;
}

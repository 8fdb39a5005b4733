// Runtime half of the C-ABI: context, one stream, stream-ordered pool, copies, module
// load / launch by name, event timer.  Replaces the cudarc calls of the reference
// (src/graph/mod.rs:152-307, src/graph/memory.rs:189-266, src/tensor.rs:145-223).
#include "runtime.h"

#include "device_utils.cuh"
#include "upload_rule.h"

#include <algorithm>
#include <atomic>
#include <thread>

int eisen_set_error(eisen_ctx* ctx, int code, const char* fmt, ...) {
    if (ctx) {
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(ctx->last_error, sizeof(ctx->last_error), fmt, ap);
        va_end(ap);
    }
    return code;
}

namespace {

// ---- copies between device memory and pinned host memory as kernels --------------------------------------------
// The runtime's own copies of 32 KB and more go through a copy engine, which a chain of kernels waits for: a kernel, such a copy and a kernel take 19.5 us where the
// copy as a kernel of one workgroup makes it 9; and an event behind a copy, recorded to know when its staging memory is free, is 3 us of
// the stream.  So an upload of up to kCopyKernelBytes is one workgroup here, and says itself that it is done.  The runtime's copy / this, in us, a kernel, the upload and a kernel in
// a row | uploads alone in a row: 32 KB 27 / 14 | 15 / 6, 64 KB 28 / 16 | 15 / 9, 96 KB 29 / 20 | 16 / 13; beyond the line 128 KB 30 / 23 | 17 / 16 but one upload, a kernel and the wait
// for them 29 / 32, 192 KB 31 / 30 | 18 / 22, 256 KB 32 / 36 | 20 / 29: one workgroup reads 9 GB/s from the host.  (Not the tickets of eisen_hip_dtoh_begin: a
// few bytes, where making them visible to the host writes the caches back: 1 us more than the event.)
constexpr int kCopyThreads = 1024;

template <typename T>
__device__ __forceinline__ void copy_by_workgroup(const T* __restrict__ src, T* __restrict__ dst, unsigned n) {
    constexpr int U = 4;
    for (unsigned i = threadIdx.x; i < n; i += U * kCopyThreads) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i + u * kCopyThreads < n) v[u] = src[i + u * kCopyThreads];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i + u * kCopyThreads < n) dst[i + u * kCopyThreads] = v[u];
    }
}
// The word says that the staging memory has been read (a thread that stores has what it read).
template <typename T>
__global__ __launch_bounds__(kCopyThreads) void copy_in_kernel(const T* __restrict__ src, T* __restrict__ dst, unsigned n, unsigned* word, unsigned number) {
    copy_by_workgroup(src, dst, n);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(word, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// f32 values to a tensor of T and, if asked for, as int32 beside it (token ids: what the lookup reads).  dst and ids begin 16 bytes aligned.
// What bounds it is the latency of the host's memory, so one launch instead of three (the values, their rounding, the ids: 5 + 3 + 5 us): training steps, three launches / one, six
// processes each, us: 8 micro-batches of 1024 tokens, hidden 1024, 10444 / 10366 (a side's runs within 20), one of 2048, hidden 256, 384 / 376, one of 1351, hidden 288, 593 / 585, of 4096
// in f32, where nothing is rounded, 2417 / 2411; of 64 in f32 261 / 258, within what runs differ by.
template <typename T>
__global__ __launch_bounds__(kCopyThreads) void copy_in_values_kernel(const float* __restrict__ src, T* __restrict__ dst, int* __restrict__ ids, unsigned n, unsigned* word,
                                                                      unsigned number) {
    constexpr int U = 4;
    typedef T T4 __attribute__((ext_vector_type(4)));
    const unsigned quads = n / 4;
    for (unsigned i = threadIdx.x; i < quads; i += U * kCopyThreads) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i + u * kCopyThreads < quads) v[u] = reinterpret_cast<const float4*>(src)[i + u * kCopyThreads];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned at = i + u * kCopyThreads;
            if (at >= quads) continue;
            T4 o;
            o[0] = from_f32<T>(v[u].x); o[1] = from_f32<T>(v[u].y); o[2] = from_f32<T>(v[u].z); o[3] = from_f32<T>(v[u].w);
            reinterpret_cast<T4*>(dst)[at] = o;
            if (ids) reinterpret_cast<int4*>(ids)[at] = make_int4((int)v[u].x, (int)v[u].y, (int)v[u].z, (int)v[u].w);
        }
    }
    if (threadIdx.x < n % 4) {
        const unsigned at = quads * 4 + threadIdx.x;
        const float v = src[at];
        dst[at] = from_f32<T>(v);
        if (ids) ids[at] = (int)v;
    }
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(word, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// A read-back in pieces: kBackGroup workgroups bring each piece, two groups in turn, and every workgroup has a word per piece, so that the host takes a piece while the
// next ones travel.
constexpr size_t kBackPiece = size_t(256) << 10, kBackRing = size_t(8) << 20;
constexpr int kBackGroup = 8, kBackPieces = (int)(kBackRing / kBackPiece), kBackWords = kBackPieces * kBackGroup;
__global__ __launch_bounds__(kCopyThreads) void read_back_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, unsigned n, unsigned* words, unsigned number) {
    constexpr unsigned PIECE = (unsigned)(kBackPiece / 16), SHARE = PIECE / kBackGroup;
    const unsigned member = blockIdx.x % kBackGroup;
    for (unsigned piece = blockIdx.x / kBackGroup; piece * PIECE < n; piece += 2) {
        const unsigned at = piece * PIECE + member * SHARE;
        if (at < n) copy_by_workgroup(src + at, dst + at, min(SHARE, n - at));
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(words + piece * kBackGroup + member, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Waits until a kernel of `stream` has set the word; a stream that has run dry or failed ends the wait as well.
int wait_word(eisen_ctx* ctx, const unsigned* word, unsigned number, hipStream_t stream) {
    for (unsigned spin = 0; __atomic_load_n(word, __ATOMIC_ACQUIRE) != number; spin++) {
        if (spin < 20000) {
            __builtin_ia32_pause();
            continue;
        }
        if (spin % 4096 != 0) {
            std::this_thread::yield();
            continue;
        }
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;  // a stream under capture cannot be asked; the word comes from before the capture
        EISEN_HIP_TRY(ctx, hipStreamIsCapturing(stream, &capture));
        if (capture != hipStreamCaptureStatusNone) continue;
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // (asking a stream ends a capture in another mode)
        EISEN_HIP_TRY(ctx, hipThreadExchangeStreamCaptureMode(&mode));
        const hipError_t q = hipStreamQuery(stream);
        EISEN_HIP_TRY(ctx, hipThreadExchangeStreamCaptureMode(&mode));
        if (q == hipSuccess) break;
        (void)hipGetLastError();
        if (q != hipErrorNotReady) EISEN_HIP_TRY(ctx, q);
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return 0;
}
// Until the slot's copy is done.
int wait_slot(eisen_ctx* ctx, eisen_ctx::StageSlot& s) {
    if (s.by_word) return wait_word(ctx, s.word, s.number, s.stream);
    EISEN_HIP_TRY(ctx, hipEventSynchronize(s.done));
    return 0;
}
// Under capture no kernel uploads: a replay would set the word again.
bool stream_captures(eisen_ctx* ctx) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(ctx->stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone;
}
// The slot's memory to the device by a kernel, where size and alignment let it; false: not.
bool upload_by_kernel(eisen_ctx* ctx, eisen_ctx::StageSlot& s, void* dst, size_t bytes) {
    if (bytes > kCopyKernelBytes || bytes % 4 != 0 || !eisen_aligned(dst, 4) || stream_captures(ctx)) return false;
    s.number++;
    if (bytes % 16 == 0 && eisen_aligned(dst, 16))
        copy_in_kernel<<<1, kCopyThreads, 0, ctx->stream>>>(static_cast<const uint4*>(s.ptr), static_cast<uint4*>(dst), (unsigned)(bytes / 16), s.word, s.number);
    else
        copy_in_kernel<<<1, kCopyThreads, 0, ctx->stream>>>(static_cast<const unsigned*>(s.ptr), static_cast<unsigned*>(dst), (unsigned)(bytes / 4), s.word, s.number);
    s.stream = ctx->stream;
    s.by_word = true;
    return true;
}

}  // namespace

extern "C" const char* eisen_hip_last_error(eisen_ctx* ctx) { return ctx ? ctx->last_error : "null context"; }

extern "C" int eisen_hip_init(int device, eisen_ctx** out) {
    if (!out) return EISEN_E_ARG;
    *out = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess) return (int)e;
    if (device < 0 || device >= count) return EISEN_E_ARG;
    e = hipSetDevice(device);
    if (e != hipSuccess) return (int)e;
    eisen_ctx* ctx = new eisen_ctx();
    ctx->device = device;
    // default priority, non-blocking with respect to the legacy null stream
    e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking);
    ctx->main_stream = ctx->stream;
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&ctx->side_stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ctx->ev_side, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ctx->ev_mark, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev_start);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev_stop);
    if (e == hipSuccess) {
        // keep freed blocks inside the driver pool instead of returning them to the OS
        hipMemPool_t pool;
        if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess) {
            uint64_t threshold = UINT64_MAX;
            (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &threshold);
        }
        (void)hipGetLastError();
    }
    if (e != hipSuccess) {
        delete ctx;
        return (int)e;
    }
    const int rc = eisen_attention_scratch_init(ctx);
    if (rc != 0) {
        (void)eisen_hip_destroy(ctx);
        return rc;
    }
    *out = ctx;
    return 0;
}

extern "C" int eisen_hip_pool_trim(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    EISEN_HIP_TRY(ctx, hipSetDevice(ctx->device));
    // every block leaves the lists before it is freed, so a failing hipFreeAsync cannot leave a freed pointer behind
    hipError_t first = hipSuccess;
    for (auto& kv : ctx->free_lists) {
        while (!kv.second.empty()) {
            void* p = kv.second.back();
            kv.second.pop_back();
            ctx->cached_bytes -= kv.first;
            const hipError_t e = hipFreeAsync(p, ctx->stream);
            if (e != hipSuccess && first == hipSuccess) first = e;
        }
    }
    ctx->free_lists.clear();
    ctx->cached_bytes = 0;
    if (first != hipSuccess) {
        (void)hipGetLastError();
        return eisen_set_error(ctx, (int)first, "eisen_hip_pool_trim: hipFreeAsync failed: %s", hipGetErrorString(first));
    }
    return 0;
}

extern "C" int eisen_hip_destroy(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    (void)hipSetDevice(ctx->device);
    ctx->stream = ctx->main_stream;
    (void)hipStreamSynchronize(ctx->side_stream);
    (void)hipStreamSynchronize(ctx->stream);
    (void)eisen_hip_pool_trim(ctx);
    for (auto& kv : ctx->live) (void)hipFreeAsync(kv.first, ctx->stream);
    for (auto& t : ctx->rope_tables) (void)hipFreeAsync(t.cos_sin, ctx->stream);
    if (ctx->ws) (void)hipFreeAsync(ctx->ws, ctx->stream);
    if (ctx->ws_side) (void)hipFreeAsync(ctx->ws_side, ctx->side_stream);
    (void)hipStreamSynchronize(ctx->side_stream);
    (void)hipStreamSynchronize(ctx->stream);
    for (auto& sl : ctx->stage) {
        if (sl.ptr) (void)hipHostFree(sl.ptr);
        if (sl.done) (void)hipEventDestroy(sl.done);
    }
    if (ctx->back) (void)hipHostFree(ctx->back);
    if (ctx->words) (void)hipHostFree(ctx->words);
    for (hipEvent_t e : ctx->prof.pool) (void)hipEventDestroy(e);
    (void)hipEventDestroy(ctx->ev_start);
    (void)hipEventDestroy(ctx->ev_stop);
    (void)hipEventDestroy(ctx->ev_fork);
    (void)hipEventDestroy(ctx->ev_side);
    (void)hipEventDestroy(ctx->ev_mark);
    (void)hipStreamDestroy(ctx->side_stream);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return 0;
}

// Work issued between side_begin and side_end runs on a second stream, after everything issued before side_begin and
// concurrently with what the main stream is given next; side_wait makes the main stream wait for it.
extern "C" int eisen_hip_side_begin(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, !ctx->side_active && !ctx->side_inline, EISEN_E_ARG, "eisen_hip_side_begin: already on the side stream");
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    EISEN_HIP_TRY(ctx, hipStreamIsCapturing(ctx->main_stream, &capture));
    EISEN_HIP_TRY(ctx, hipEventRecord(ctx->ev_fork, ctx->main_stream));
    ctx->mark = capture == hipStreamCaptureStatusNone ? ctx->ev_fork : nullptr;  // (an event recorded in a capture cannot be asked)
    EISEN_HIP_TRY(ctx, hipStreamWaitEvent(ctx->side_stream, ctx->ev_fork, 0));
    ctx->stream = ctx->side_stream;
    ctx->side_active = true;
    return 0;
}
// A wait of one stream for another costs the host 14 us, five launches: where the device has caught up with the host, as in steps of
// many short kernels, work beside the chain gains nothing and the fork delays everything behind it.  Caught up: what the main stream was
// given before the last fork, or the last call of this function, is done.  A step of hidden 288, 4 layers and 1351 tokens, whose kernels take 715 us
// and whose host work took 800 with 15 waits: 822 -> 786 us; the ~14 M model's 8192 tokens, where the device is behind and the work
// beside the chain is worth 0.3 to 1.3 %: the same.
extern "C" int eisen_hip_side_begin_if_behind(eisen_ctx* ctx, int* forked) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, forked != nullptr, EISEN_E_ARG, "eisen_hip_side_begin_if_behind: forked is null");
    EISEN_REQUIRE(ctx, !ctx->side_active && !ctx->side_inline, EISEN_E_ARG, "eisen_hip_side_begin_if_behind: already on the side stream");
    *forked = 1;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    EISEN_HIP_TRY(ctx, hipStreamIsCapturing(ctx->main_stream, &capture));
    if (capture == hipStreamCaptureStatusNone) {  // (events outside a capture are not asked for inside one)
        hipError_t q = hipErrorNotReady;
        if (ctx->mark) {  // (asking an event ends a capture that this or another thread has begun on any stream, unless the thread is in relaxed mode)
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
            EISEN_HIP_TRY(ctx, hipThreadExchangeStreamCaptureMode(&mode));
            q = hipEventQuery(ctx->mark);
            EISEN_HIP_TRY(ctx, hipThreadExchangeStreamCaptureMode(&mode));
        }
        if (q != hipSuccess) (void)hipGetLastError();  // not ready is an answer, not an error for the next launch check to find
        if (q != hipSuccess && q != hipErrorNotReady) EISEN_HIP_TRY(ctx, q);
        if (q == hipSuccess) {
            // (a record is a packet between two kernels: one more beside each of the 19 forks cost the ~14 M model's step 4 %, so a fork's own serves)
            EISEN_HIP_TRY(ctx, hipEventRecord(ctx->ev_mark, ctx->main_stream));
            ctx->mark = ctx->ev_mark;
            ctx->side_inline = true;
            *forked = 0;
            return 0;
        }
    }
    return eisen_hip_side_begin(ctx);
}
extern "C" int eisen_hip_side_end(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    if (ctx->side_inline) {
        ctx->side_inline = false;
        return 0;
    }
    EISEN_REQUIRE(ctx, ctx->side_active, EISEN_E_ARG, "eisen_hip_side_end: not on the side stream");
    ctx->stream = ctx->main_stream;
    ctx->side_active = false;
    EISEN_HIP_TRY(ctx, hipEventRecord(ctx->ev_side, ctx->side_stream));
    ctx->side_pending = true;
    return 0;
}
extern "C" int eisen_hip_side_wait(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, !ctx->side_active && !ctx->side_inline, EISEN_E_ARG, "eisen_hip_side_wait: still on the side stream");
    if (ctx->side_pending) EISEN_HIP_TRY(ctx, hipStreamWaitEvent(ctx->main_stream, ctx->ev_side, 0));
    ctx->side_pending = false;
    return 0;
}

extern "C" int eisen_hip_stream_sync(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    if (ctx->side_pending || ctx->side_active) EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->side_stream));
    EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->main_stream));
    ctx->waited = true;
    return 0;
}

extern "C" void* eisen_hip_stream(eisen_ctx* ctx) { return ctx ? (void*)ctx->stream : nullptr; }

extern "C" int eisen_hip_malloc(eisen_ctx* ctx, size_t bytes, void** out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, out != nullptr, EISEN_E_ARG, "eisen_hip_malloc: out is null");
    if (bytes == 0) bytes = 4;
    bytes = (bytes + 255) & ~size_t(255);  // 256-byte granules keep every block 16-byte aligned
    void* p = nullptr;
    auto it = ctx->free_lists.find(bytes);
    if (it != ctx->free_lists.end() && !it->second.empty()) {
        p = it->second.back();
        it->second.pop_back();
        ctx->cached_bytes -= bytes;
    } else {
        ctx->driver_allocs++;
        hipError_t e = hipMallocAsync(&p, bytes, ctx->stream);
        if (e != hipSuccess) {
            // out of memory: give cached blocks back and retry once
            (void)hipGetLastError();
            (void)eisen_hip_pool_trim(ctx);
            (void)hipStreamSynchronize(ctx->stream);
            e = hipMallocAsync(&p, bytes, ctx->stream);
            if (e != hipSuccess)
                return eisen_set_error(ctx, (int)e, "hipMallocAsync(%zu bytes) failed: %s", bytes,
                                       hipGetErrorString(e));
        }
    }
    ctx->live[p] = bytes;
    ctx->in_use_bytes += bytes;
    if (ctx->in_use_bytes > ctx->peak_in_use_bytes) ctx->peak_in_use_bytes = ctx->in_use_bytes;
    *out = p;
    return 0;
}

extern "C" int eisen_hip_malloc_zeroed(eisen_ctx* ctx, size_t bytes, void** out) {
    int rc = eisen_hip_malloc(ctx, bytes, out);
    if (rc) return rc;
    return eisen_hip_memset_zero(ctx, *out, ctx->live[*out]);
}

extern "C" int eisen_hip_free(eisen_ctx* ctx, void* ptr) {
    EISEN_CHECK_CTX(ctx);
    if (!ptr) return 0;
    auto it = ctx->live.find(ptr);
    EISEN_REQUIRE(ctx, it != ctx->live.end(), EISEN_E_ARG, "eisen_hip_free: %p was not allocated by this context", ptr);
    const size_t bytes = it->second;
    ctx->live.erase(it);
    ctx->in_use_bytes -= bytes;
    ctx->free_lists[bytes].push_back(ptr);
    ctx->cached_bytes += bytes;
    return 0;
}

extern "C" int eisen_hip_pool_peak(eisen_ctx* ctx, size_t* peak_in_use_bytes, int reset) {
    EISEN_CHECK_CTX(ctx);
    if (peak_in_use_bytes) *peak_in_use_bytes = ctx->peak_in_use_bytes;
    if (reset) ctx->peak_in_use_bytes = ctx->in_use_bytes;
    return 0;
}

extern "C" int eisen_hip_mem_info(eisen_ctx* ctx, size_t* free_bytes, size_t* total_bytes) {
    EISEN_CHECK_CTX(ctx);
    size_t f = 0, t = 0;
    EISEN_HIP_TRY(ctx, hipMemGetInfo(&f, &t));
    if (free_bytes) *free_bytes = f;
    if (total_bytes) *total_bytes = t;
    return 0;
}

extern "C" int eisen_hip_driver_allocs(eisen_ctx* ctx, size_t* count_out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, count_out != nullptr, EISEN_E_ARG, "driver_allocs: count_out is null");
    *count_out = ctx->driver_allocs;
    return 0;
}

extern "C" int eisen_hip_pool_stats(eisen_ctx* ctx, size_t* in_use_bytes, size_t* cached_bytes) {
    EISEN_CHECK_CTX(ctx);
    if (in_use_bytes) *in_use_bytes = ctx->in_use_bytes;
    if (cached_bytes) *cached_bytes = ctx->cached_bytes;
    return 0;
}

// A block of the driver's pool on the active stream.  Out of memory: what the free lists hold is given back and the request repeated once.
static int driver_alloc(eisen_ctx* ctx, size_t bytes, const char* what, void** out) {
    ctx->driver_allocs++;
    hipError_t e = hipMallocAsync(out, bytes, ctx->stream);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        (void)hipStreamSynchronize(ctx->main_stream);  // the lists' blocks may still be in use on either stream
        (void)hipStreamSynchronize(ctx->side_stream);
        (void)eisen_hip_pool_trim(ctx);
        (void)hipStreamSynchronize(ctx->stream);
        e = hipMallocAsync(out, bytes, ctx->stream);
    }
    if (e != hipSuccess) {
        *out = nullptr;
        return eisen_set_error(ctx, EISEN_E_NOMEM, "%s of %zu bytes: %s", what, bytes, hipGetErrorString(e));
    }
    return 0;
}

int EisenScratch::get(eisen_ctx* ctx, size_t bytes) {
    if (bytes <= kWorkspaceKeep) return eisen_workspace(ctx, bytes, &ptr);
    const int rc = driver_alloc(ctx, bytes, "scratch", &own);
    if (rc) return rc;
    stream = ctx->stream;
    ptr = own;
    return 0;
}
EisenScratch::~EisenScratch() {
    if (own) (void)hipFreeAsync(own, stream);
}

int eisen_workspace(eisen_ctx* ctx, size_t bytes, void** out) {
    // one block per stream: each is allocated, used and freed in the order of its own stream
    void*& ws = ctx->side_active ? ctx->ws_side : ctx->ws;
    size_t& ws_bytes = ctx->side_active ? ctx->ws_side_bytes : ctx->ws_bytes;
    if (bytes > ws_bytes) {
        // stream order makes the old block safe to free while earlier kernels still read it
        if (ws) EISEN_HIP_TRY(ctx, hipFreeAsync(ws, ctx->stream));
        ws = nullptr;
        ws_bytes = 0;
        size_t want = (bytes + (size_t(1) << 20) - 1) & ~((size_t(1) << 20) - 1);
        const int rc = driver_alloc(ctx, want, "workspace", &ws);
        if (rc) return rc;
        ws_bytes = want;
    }
    *out = ws;
    return 0;
}

// the pinned words: 64 bytes per slot, then a read-back's
static int eisen_words(eisen_ctx* ctx) {
    if (ctx->words) return 0;
    ctx->driver_allocs++;
    const size_t bytes = 64 * (size_t)eisen_ctx::kStageSlots + sizeof(unsigned) * (size_t)kBackWords;
    EISEN_HIP_TRY(ctx, hipHostMalloc(reinterpret_cast<void**>(&ctx->words), bytes, hipHostMallocDefault));
    memset(ctx->words, 0, bytes);
    return 0;
}

int eisen_staging(eisen_ctx* ctx, size_t bytes, eisen_ctx::StageSlot** out) {
    int tries = 0;
    while (ctx->stage[ctx->stage_next].reserved && tries < eisen_ctx::kStageSlots) {
        ctx->stage_next = (ctx->stage_next + 1) % eisen_ctx::kStageSlots;
        tries++;
    }
    EISEN_REQUIRE(ctx, tries < eisen_ctx::kStageSlots, EISEN_E_STATE, "every staging slot holds an uncollected eisen_hip_dtoh_begin result");
    eisen_ctx::StageSlot& s = ctx->stage[ctx->stage_next];
    ctx->stage_next = (ctx->stage_next + 1) % eisen_ctx::kStageSlots;
    if (!s.done) EISEN_HIP_TRY(ctx, hipEventCreateWithFlags(&s.done, hipEventDisableTiming));
    if (!s.word) {
        const int rc = eisen_words(ctx);
        if (rc) return rc;
        s.word = ctx->words + 16 * (&s - ctx->stage);
    }
    if (s.in_flight) {
        const int rc = wait_slot(ctx, s);
        if (rc) return rc;
        s.in_flight = false;
    }
    s.by_word = false;
    if (bytes > s.bytes) {
        if (s.ptr) EISEN_HIP_TRY(ctx, hipHostFree(s.ptr));
        s.ptr = nullptr;
        s.bytes = 0;
        size_t want = (bytes + (size_t(1) << 16) - 1) & ~((size_t(1) << 16) - 1);
        ctx->driver_allocs++;
        EISEN_HIP_TRY(ctx, hipHostMalloc(&s.ptr, want, hipHostMallocDefault));
        s.bytes = want;
    }
    *out = &s;
    return 0;
}

static constexpr size_t kStageLimit = size_t(8) << 20;

extern "C" int eisen_hip_htod(eisen_ctx* ctx, void* dst, const void* src, size_t bytes) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst && src, EISEN_E_ARG, "eisen_hip_htod: null pointer");
    if (bytes == 0) return 0;
    if (bytes <= kStageLimit) {
        // small uploads (token ids, targets, tables) go through pinned staging and stay asynchronous
        eisen_ctx::StageSlot* st = nullptr;
        int rc = eisen_staging(ctx, bytes, &st);
        if (rc) return rc;
        memcpy(st->ptr, src, bytes);
        if (upload_by_kernel(ctx, *st, dst, bytes)) {
            EISEN_LAUNCH_CHECK(ctx, "eisen_hip_htod");
        } else {
            EISEN_HIP_TRY(ctx, hipMemcpyAsync(dst, st->ptr, bytes, hipMemcpyHostToDevice, ctx->stream));
            EISEN_HIP_TRY(ctx, hipEventRecord(st->done, ctx->stream));
        }
        st->in_flight = true;
        return 0;
    }
    EISEN_HIP_TRY(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

extern "C" int eisen_hip_htod_values(eisen_ctx* ctx, void* dst, int dtype, int32_t* ids, const float* src, size_t n) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst && src, EISEN_E_ARG, "eisen_hip_htod_values: null pointer");
    EISEN_REQUIRE(ctx, eisen_dtype_ok(dtype), EISEN_E_ARG, "eisen_hip_htod_values: unknown dtype %d", dtype);
    if (n == 0) return 0;
    if (n <= kCopyKernelBytes / sizeof(float) && eisen_aligned(dst, 16) && eisen_aligned(ids, 16) && !stream_captures(ctx)) {
        eisen_ctx::StageSlot* st = nullptr;
        const int rc = eisen_staging(ctx, n * sizeof(float), &st);
        if (rc) return rc;
        memcpy(st->ptr, src, n * sizeof(float));
        st->number++;
        const float* from = static_cast<const float*>(st->ptr);
        EisenProfScope prof(ctx, "htod_values", (double)n * (4.0 + eisen_dtype_size(dtype) + (ids ? 4.0 : 0.0)));
        if (dtype == EISEN_F32) copy_in_values_kernel<float><<<1, kCopyThreads, 0, ctx->stream>>>(from, static_cast<float*>(dst), ids, (unsigned)n, st->word, st->number);
        else copy_in_values_kernel<bf16_t><<<1, kCopyThreads, 0, ctx->stream>>>(from, static_cast<bf16_t*>(dst), ids, (unsigned)n, st->word, st->number);
        st->stream = ctx->stream;
        st->by_word = true;
        EISEN_LAUNCH_CHECK(ctx, "eisen_hip_htod_values");
        st->in_flight = true;
        return 0;
    }
    int rc = 0;
    if (dtype == EISEN_F32) {
        rc = eisen_hip_htod(ctx, dst, src, n * sizeof(float));
    } else {
        void* tmp = nullptr;
        rc = eisen_hip_malloc(ctx, n * sizeof(float), &tmp);
        if (rc) return rc;
        rc = eisen_hip_htod(ctx, tmp, src, n * sizeof(float));
        if (!rc) rc = eisen_hip_cast(ctx, tmp, EISEN_F32, dst, EISEN_BF16, n);
        const int rc_free = eisen_hip_free(ctx, tmp);
        if (!rc) rc = rc_free;
    }
    if (rc || !ids) return rc;
    std::vector<int32_t> whole(n);
    for (size_t i = 0; i < n; i++) whole[i] = src[i] >= -2147483648.0f && src[i] < 2147483648.0f ? (int32_t)src[i] : 0;
    return eisen_hip_htod(ctx, ids, whole.data(), n * sizeof(int32_t));
}

// Memory that the device writes itself (pinned).
static bool known_to_device(const void* p) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}
// Device memory into the caller's, as it is or (widen) bf16 as f32.  Through pinned memory in pieces (read_back_kernel); what is small, not aligned or under capture
// goes by the runtime's copy.  That copy and this behind a kernel, in us: 4 KB 24 and 25 (the line is at 16 KB, where they part), 64 KB 28 and 24, 256 KB 37 and 30, 1 MB 78
// and 54, 4 MB 264 and 129; 512 MB 32100 and 24900.  A forward pass with its 201 x 8192 bf16 logits read back 579 and 369.
// The runtime's copy also where it is ahead: into pinned memory (64 KB 10 and 19, 1 MB 27 and 48, 64 MB 1185 and 2370), and above 16 KB (up to which it is 24 and this 19) to 1 MB where its
// copy engine has no kernel to wait for (20 KB 11 and 18, 64 KB 12 and 19, 256 KB 20 and 25, 512 KB 31 and 36, 1 MB 60 and 49); to be widened, there, into the ring (20 KB of bf16 11 and
// 19, 64 KB 15 and 21, 128 KB 19 and 28, 256 KB 28 and 35, 512 KB 44 and 46).
static int read_back(eisen_ctx* ctx, void* dst, const void* src, size_t bytes, bool widen) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    EISEN_HIP_TRY(ctx, hipStreamIsCapturing(ctx->stream, &capture));
    const size_t whole = bytes / 16 * 16;
    char* out = static_cast<char*>(dst);
    auto take = [&](const void* from, size_t n) {
        if (widen) {
            const uint16_t* __restrict__ f = static_cast<const uint16_t*>(from);
            uint32_t* __restrict__ t = reinterpret_cast<uint32_t*>(out);
            for (size_t i = 0; i < n / 2; i++) t[i] = (uint32_t)f[i] << 16;
        } else {
            memcpy(out, from, n);
        }
        out += widen ? 2 * n : n;
    };
    size_t done = 0;
    bool ring = whole >= (size_t(16) << 10) && eisen_aligned(src, 16) && capture == hipStreamCaptureStatusNone;
    const bool on_main = ctx->stream == ctx->main_stream, idle = ctx->waited && on_main;
    if (ring && !widen) ring = !known_to_device(dst) && !(idle && whole > (size_t(16) << 10) && whole < (size_t(1) << 20));
    if (ring) {
        const int rc = eisen_words(ctx);
        if (rc) return rc;
        const size_t want = (std::min(whole, kBackRing) + kBackPiece - 1) / kBackPiece * kBackPiece;
        if (ctx->back_bytes < want) {
            if (ctx->back) EISEN_HIP_TRY(ctx, hipHostFree(ctx->back));
            ctx->back = nullptr;
            ctx->back_bytes = 0;
            ctx->driver_allocs++;
            EISEN_HIP_TRY(ctx, hipHostMalloc(&ctx->back, want, hipHostMallocDefault));
            ctx->back_bytes = want;
        }
        if (widen && idle && whole > (size_t(16) << 10) && whole < (size_t(512) << 10)) {
            EISEN_HIP_TRY(ctx, hipMemcpyAsync(ctx->back, src, whole, hipMemcpyDeviceToHost, ctx->stream));
            EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
            take(ctx->back, whole);
            done = whole;
        }
        unsigned* words = ctx->words + 16 * eisen_ctx::kStageSlots;
        while (done < whole) {
            const size_t n = std::min(whole - done, ctx->back_bytes);
            const unsigned number = ++ctx->back_number;
            read_back_kernel<<<2 * kBackGroup, kCopyThreads, 0, ctx->stream>>>(reinterpret_cast<const uint4*>(static_cast<const char*>(src) + done), static_cast<uint4*>(ctx->back),
                                                                              (unsigned)(n / 16), words, number);
            EISEN_LAUNCH_CHECK(ctx, "eisen_hip_dtoh");
            for (size_t at = 0, piece = 0; at < n; at += kBackPiece, piece++) {
                for (int w = 0; w < kBackGroup; w++) {
                    const int rw = wait_word(ctx, words + piece * kBackGroup + w, number, ctx->stream);
                    if (rw) return rw;
                }
                take(static_cast<char*>(ctx->back) + at, std::min(kBackPiece, n - at));
            }
            done += n;
        }
    }
    if (on_main) ctx->waited = true;
    if (done == bytes) return 0;
    const size_t left = bytes - done;
    char* raw = widen ? out + left : out;  // (in the upper half of what is to hold it as f32: element i is read before any write reaches it)
    EISEN_HIP_TRY(ctx, hipMemcpyAsync(raw, static_cast<const char*>(src) + done, left, hipMemcpyDeviceToHost, ctx->stream));
    EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    for (size_t i = 0; widen && i < left / 2; i++) {
        uint16_t half;
        memcpy(&half, raw + 2 * i, 2);
        const uint32_t value = (uint32_t)half << 16;
        memcpy(out + 4 * i, &value, 4);
    }
    return 0;
}

extern "C" int eisen_hip_dtoh(eisen_ctx* ctx, void* dst, const void* src, size_t bytes) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst && src, EISEN_E_ARG, "eisen_hip_dtoh: null pointer");
    if (bytes == 0) return 0;
    return read_back(ctx, dst, src, bytes, false);
}

extern "C" int eisen_hip_dtoh_widen(eisen_ctx* ctx, float* dst, const void* src_bf16, size_t n) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst && src_bf16, EISEN_E_ARG, "eisen_hip_dtoh_widen: null pointer");
    if (n == 0) return 0;
    return read_back(ctx, dst, src_bf16, 2 * n, true);
}

extern "C" int eisen_hip_dtoh_begin(eisen_ctx* ctx, const void* src, size_t bytes, int* ticket_out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, src && ticket_out, EISEN_E_ARG, "eisen_hip_dtoh_begin: null pointer");
    EISEN_REQUIRE(ctx, bytes > 0 && bytes <= kStageLimit, EISEN_E_SHAPE, "eisen_hip_dtoh_begin: %zu bytes (1 .. %zu supported)", bytes, kStageLimit);
    int reserved = 0;
    for (const auto& sl : ctx->stage) reserved += sl.reserved ? 1 : 0;
    EISEN_REQUIRE(ctx, reserved < eisen_ctx::kStageSlots / 2, EISEN_E_STATE, "eisen_hip_dtoh_begin: %d copies not collected yet", reserved);
    eisen_ctx::StageSlot* st = nullptr;
    int rc = eisen_staging(ctx, bytes, &st);
    if (rc) return rc;
    EISEN_HIP_TRY(ctx, hipMemcpyAsync(st->ptr, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    EISEN_HIP_TRY(ctx, hipEventRecord(st->done, ctx->stream));
    st->in_flight = true;
    st->reserved = true;
    *ticket_out = (int)(st - ctx->stage);
    return 0;
}

extern "C" int eisen_hip_dtoh_finish(eisen_ctx* ctx, int ticket, void* dst, size_t bytes) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst != nullptr, EISEN_E_ARG, "eisen_hip_dtoh_finish: null pointer");
    EISEN_REQUIRE(ctx, ticket >= 0 && ticket < eisen_ctx::kStageSlots && ctx->stage[ticket].reserved, EISEN_E_STATE,
                  "eisen_hip_dtoh_finish: ticket %d names no pending copy", ticket);
    eisen_ctx::StageSlot& s = ctx->stage[ticket];
    EISEN_REQUIRE(ctx, bytes <= s.bytes, EISEN_E_ARG, "eisen_hip_dtoh_finish: %zu bytes asked of a %zu-byte slot", bytes, s.bytes);
    s.reserved = false;
    const int rc = wait_slot(ctx, s);  // for this copy only: later work stays queued
    if (rc) return rc;
    s.in_flight = false;
    memcpy(dst, s.ptr, bytes);
    return 0;
}

extern "C" int eisen_hip_dtod(eisen_ctx* ctx, void* dst, const void* src, size_t bytes) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst && src, EISEN_E_ARG, "eisen_hip_dtod: null pointer");
    if (bytes == 0) return 0;
    EISEN_HIP_TRY(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
    ctx->waited = false;
    return 0;
}

extern "C" int eisen_hip_memset_zero(eisen_ctx* ctx, void* dst, size_t bytes) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, dst != nullptr, EISEN_E_ARG, "eisen_hip_memset_zero: null pointer");
    if (bytes == 0) return 0;
    // a fill kernel, not hipMemsetAsync: a memset node recorded into a captured graph has replayed wrongly on this
    // hardware generation, and callers may capture the step
    if (bytes % 4 == 0 && eisen_aligned(dst, 4)) return eisen_hip_fill(ctx, dst, EISEN_F32, 0.0f, bytes / 4);
    EISEN_HIP_TRY(ctx, hipMemsetAsync(dst, 0, bytes, ctx->stream));
    return 0;
}

extern "C" int eisen_hip_module_load(eisen_ctx* ctx, const void* image, size_t len, eisen_module** out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, image && len && out, EISEN_E_ARG, "eisen_hip_module_load: null image or out");
    hipModule_t mod;
    EISEN_HIP_TRY(ctx, hipModuleLoadData(&mod, image));
    *out = new eisen_module{mod};
    return 0;
}

extern "C" int eisen_hip_module_unload(eisen_ctx* ctx, eisen_module* mod) {
    EISEN_CHECK_CTX(ctx);
    if (!mod) return 0;
    EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    EISEN_HIP_TRY(ctx, hipModuleUnload(mod->mod));
    delete mod;
    return 0;
}

extern "C" int eisen_hip_get_function(eisen_ctx* ctx, eisen_module* mod, const char* name, eisen_function** out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, mod && name && out, EISEN_E_ARG, "eisen_hip_get_function: null argument");
    hipFunction_t fn;
    hipError_t e = hipModuleGetFunction(&fn, mod->mod, name);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return eisen_set_error(ctx, (int)e, "kernel '%s' not found in module: %s", name, hipGetErrorString(e));
    }
    *out = new eisen_function{fn};  // lives as long as the process; a handful per module
    return 0;
}

extern "C" int eisen_hip_launch(eisen_ctx* ctx, eisen_function* fn, const unsigned grid[3], const unsigned block[3],
                                unsigned shared_bytes, void** args) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, fn && grid && block, EISEN_E_ARG, "eisen_hip_launch: null argument");
    EISEN_REQUIRE(ctx, grid[0] && grid[1] && grid[2] && block[0] && block[1] && block[2], EISEN_E_ARG,
                  "eisen_hip_launch: zero grid or block dimension");
    EISEN_REQUIRE(ctx, (size_t)block[0] * block[1] * block[2] <= 1024, EISEN_E_SHAPE,
                  "eisen_hip_launch: more than 1024 threads per block");
    EISEN_HIP_TRY(ctx, hipModuleLaunchKernel(fn->fn, grid[0], grid[1], grid[2], block[0], block[1], block[2],
                                             shared_bytes, ctx->stream, args, nullptr));
    ctx->waited = false;
    return 0;
}

extern "C" int eisen_hip_timer_start(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    EISEN_HIP_TRY(ctx, hipEventRecord(ctx->ev_start, ctx->stream));
    ctx->timer_running = true;
    return 0;
}

extern "C" int eisen_hip_timer_stop(eisen_ctx* ctx, float* ms_out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, ctx->timer_running, EISEN_E_STATE, "eisen_hip_timer_stop without eisen_hip_timer_start");
    EISEN_HIP_TRY(ctx, hipEventRecord(ctx->ev_stop, ctx->stream));
    EISEN_HIP_TRY(ctx, hipEventSynchronize(ctx->ev_stop));
    float ms = 0.f;
    EISEN_HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev_start, ctx->ev_stop));
    ctx->timer_running = false;
    if (ms_out) *ms_out = ms;
    return 0;
}

// ---- per-kernel timing ----------------------------------------------------------------------------

int eisen_prof_begin(eisen_ctx* ctx, const char* name, double work, bool is_flops) {
    eisen_prof& p = ctx->prof;
    int key = -1;
    for (size_t i = 0; i < p.names.size(); i++)
        if (p.names[i] == name) key = (int)i;
    if (key < 0) {
        p.names.push_back(name);
        p.is_flops.push_back(is_flops ? 1 : 0);
        key = (int)p.names.size() - 1;
    }
    while (p.pool.size() < p.pool_used + 2) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return -1;
        p.pool.push_back(e);
    }
    eisen_prof_rec r{key, p.pool[p.pool_used], p.pool[p.pool_used + 1], work};
    p.pool_used += 2;
    if (hipEventRecord(r.start, ctx->stream) != hipSuccess) return -1;
    p.recs.push_back(r);
    return (int)p.recs.size() - 1;
}
void eisen_prof_end(eisen_ctx* ctx, int rec) { (void)hipEventRecord(ctx->prof.recs[rec].stop, ctx->stream); }

extern "C" int eisen_hip_profile_start(eisen_ctx* ctx) {
    EISEN_CHECK_CTX(ctx);
    ctx->prof.enabled = true;
    ctx->prof.recs.clear();
    ctx->prof.pool_used = 0;
    return 0;
}

extern "C" int eisen_hip_profile_stop(eisen_ctx* ctx, eisen_prof_entry* out, size_t capacity, size_t* count_out) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, count_out != nullptr, EISEN_E_ARG, "eisen_hip_profile_stop: null count_out");
    eisen_prof& p = ctx->prof;
    p.enabled = false;
    // instrumented launches may sit on either stream: both have to be done before their events are read
    EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->side_stream));
    EISEN_HIP_TRY(ctx, hipStreamSynchronize(ctx->main_stream));
    std::vector<eisen_prof_entry> acc(p.names.size());
    for (size_t i = 0; i < p.names.size(); i++) {
        std::memset(&acc[i], 0, sizeof(eisen_prof_entry));
        std::strncpy(acc[i].name, p.names[i].c_str(), sizeof(acc[i].name) - 1);
        acc[i].work_is_flops = p.is_flops[i];
    }
    for (const eisen_prof_rec& r : p.recs) {
        float ms = 0.f;
        EISEN_HIP_TRY(ctx, hipEventElapsedTime(&ms, r.start, r.stop));
        acc[r.key].ms += ms;
        acc[r.key].work += r.work;
        acc[r.key].launches += 1;
    }
    size_t n = 0;
    for (const eisen_prof_entry& e : acc)
        if (e.launches) {
            if (out && n < capacity) out[n] = e;
            n++;
        }
    *count_out = n;
    p.recs.clear();
    p.pool_used = 0;
    return 0;
}

// Fused softmax-cross-entropy forward+backward: one read of the logits, one write of dLogits.
//
// One workgroup owns one row.  The row is loaded once with 16-byte packets and stays in
// registers in its storage type (VPT packets per lane) across the three phases: row max (+ first
// argmax when asked for), exponentials and their sum, gradient write (exponentials formed again).  Reductions are wave64 shuffles plus one LDS exchange
// between the block's waves.  The row is read and its gradient written with streaming (non-temporal) accesses: each byte
// is touched once, and keeping it out of the caches' way is worth 4-5 % at 8192 x 32000.  Per-row losses go to a buffer; a second one-block kernel sums
// them in a fixed order, so the loss carries no float atomics and is reproducible.
//
// Follows Graph::cross_entropy / cross_entropy_masked (src/graph/ops/reduction.rs:676-706,
// :897-931): p = exp(x - max) / sum, loss_row = -ln(p_t + 1e-8), dlogit = (p - onehot) * scale.
#include <type_traits>

#include "device_utils.cuh"
#include "runtime.h"

namespace {

struct ArgMax {
    float v;
    int i;
};
__device__ __forceinline__ ArgMax argmax_combine(ArgMax a, ArgMax b) {
    // first index of the maximum wins on ties
    if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
    return a;
}
__device__ __forceinline__ ArgMax wave_argmax(ArgMax a) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ArgMax b;
        b.v = __shfl_xor(a.v, o, 64);
        b.i = __shfl_xor(a.i, o, 64);
        a = argmax_combine(a, b);
    }
    return a;
}

// RAGGED: class counts that are no multiple of a packet.  A row then begins and ends inside a packet; the kernel works on the
// aligned packets that cover it (column -shift is the first one's first element), elements of the neighbouring rows count
// as -inf, and only the two packets at the ends are stored element by element.  8192 rows of 30001 bf16: 196 us against 676 for
// the three passes of 2-byte accesses of ce_generic_kernel.
template <typename T, int THREADS, int VPT, bool WANT_ARGMAX, bool RAGGED>
__global__ __launch_bounds__(THREADS) void ce_fused_kernel(const T* __restrict__ logits, const int32_t* __restrict__ targets,
                                                           T* __restrict__ dlogits, float* __restrict__ row_loss,
                                                           int32_t* __restrict__ argmax_out, float* __restrict__ target_logit_out,
                                                           int rows, int classes, float scale) {
    constexpr int N = Pack<T>::N;
    constexpr int W = THREADS / kWave;
    constexpr float kLog2e = 1.4426950408889634f;
    __shared__ float s_f[W];
    __shared__ int s_i[W];
    const size_t row = blockIdx.x;
    const int target = targets[row];
    const T* xr = logits + row * classes;
    T* gr = dlogits + row * classes;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    constexpr bool STREAM = !RAGGED || THREADS * VPT > 512;  // (short rows inside packets: 16000 x 1001 f32 27 us, 31 streaming)
    const int shift = RAGGED ? (int)(row * classes % N) : 0;
    auto column = [&](int v) { return (v * THREADS + (int)threadIdx.x) * N - shift; };   // of the lane's packet v
    auto store = [&](int c, const Pack<T>& g, auto streaming) {
        if (!RAGGED || (c >= 0 && c + N <= classes)) {
            if (decltype(streaming)::value) store_pack_streaming(gr + c, g);
            else store_pack(gr + c, g);
        } else {
#pragma unroll
            for (int j = 0; j < N; j++)
                if (c + j >= 0 && c + j < classes) gr[c + j] = from_f32<T>(g.get(j));
        }
    };

    // masked row: zero gradient, no loss (src/graph/ops/reduction.rs:898, :925).  A target beyond the
    // class count (the reference would panic on the index) is treated the same way: the host
    // validates targets before upload, the device only has to stay inside the row.
    if (target < 0 || target >= classes) {
        Pack<T> z;
#pragma unroll
        for (int j = 0; j < N; j++) z.set(j, 0.f);
#pragma unroll
        for (int v = 0; v < VPT; v++) {
            const int c = column(v);
            if (c < classes) store(c, z, std::false_type{});
        }
        if (threadIdx.x == 0) {
            row_loss[row] = 0.f;
            if (argmax_out) argmax_out[row] = -1;
            if (target_logit_out) target_logit_out[row] = 0.f;
        }
        return;
    }

    // phase 1: the row comes in once (VPT packets per lane, all loads in flight together) and stays in
    // registers in its storage type: half the registers of an f32 copy, so twice the workgroups per CU
    // keep loads in flight.  Running maximum (and, when asked for, its first index).
    Pack<T> raw[VPT];
    ArgMax am{-INFINITY, 0x7fffffff};
    // elements from the row's start to the end of the buffer (rows, not gridDim.x: a kernel that asks for the size of its grid gets
    // hidden arguments, and filling those in cost 0.5 us of every launch)
    const long long left = (long long)(rows - (int)row) * classes;
#pragma unroll
    for (int v = 0; v < VPT; v++) {
        const int c = column(v);
        if (c < classes && (!RAGGED || (long long)c + N <= left)) raw[v] = STREAM ? load_pack_streaming(xr + c) : load_pack(xr + c);
    }
    if constexpr (RAGGED) {  // after the loads: a second path beside each of them would make the compiler wait for it there
        if (left < classes + N) {  // (uniform) the rows whose last packet would reach past the buffer
#pragma unroll
            for (int v = 0; v < VPT; v++) {
                const int c = column(v);
                if (c < classes && (long long)c + N > left) {
#pragma unroll
                    for (int j = 0; j < N; j++) raw[v].set(j, c + j >= 0 && c + j < classes ? to_f32(xr[c + j]) : -INFINITY);
                }
            }
        }
#pragma unroll
        for (int v = 0; v < VPT; v++) {
            const int c = column(v);
            if (c < 0 || c + N > classes) {
#pragma unroll
                for (int j = 0; j < N; j++)
                    if (c + j < 0 || c + j >= classes) raw[v].set(j, -INFINITY);
            }
        }
    }
#pragma unroll
    for (int v = 0; v < VPT; v++) {
        const int c = column(v);
        if (c < classes) {
#pragma unroll
            for (int j = 0; j < N; j++) {
                const float xv = raw[v].get(j);
                if (WANT_ARGMAX) {
                    if (xv > am.v) {  // ascending c within the lane: strict > keeps the first
                        am.v = xv;
                        am.i = c + j;
                    }
                } else {
                    am.v = fmaxf(am.v, xv);
                }
            }
        }
    }
    if (WANT_ARGMAX) {
        am = wave_argmax(am);
        if (W > 1) {
            if (lane == 0) {
                s_f[wid] = am.v;
                s_i[wid] = am.i;
            }
            __syncthreads();
            am = ArgMax{s_f[0], s_i[0]};
#pragma unroll
            for (int k = 1; k < W; k++) am = argmax_combine(am, ArgMax{s_f[k], s_i[k]});
            __syncthreads();
        }
    } else {
        am.v = block_max<THREADS>(am.v, s_f);
    }
    const float mx = am.v;

    // phase 2: row sum of e = 2^(x*log2e - max*log2e).  The exponent is never positive, so the bare
    // hardware exp2 (results below 2^-126 flush to zero) is exact enough.  The variants that took over from
    // ce_generic_kernel subtract first, as it does: a row of nothing but the type's lowest value stays finite.
    constexpr bool SUBTRACT = RAGGED || VPT > 8;
    const float bias = -mx * kLog2e;
    float mx_now = mx;
    auto exponential = [&](float x) { return __builtin_amdgcn_exp2f(SUBTRACT ? (x - mx_now) * kLog2e : fmaf(x, kLog2e, bias)); };
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < VPT; v++) {
        const int c = column(v);
        if (c < classes) {
#pragma unroll
            for (int j = 0; j < N; j++) sum += exponential(raw[v].get(j));
        }
    }
    sum = block_sum<THREADS>(sum, s_f);
    if (VPT > 8) asm volatile("" : "+v"(mx_now));
    const float inv = 1.0f / sum;
    const float gscale = inv * scale;

    // phase 3: dlogit = (e/sum - onehot) * scale with e recomputed (a second exp2 costs less than the
    // registers that keeping it would take: at 16 packets the compiler would keep it, in scratch); the lane that holds the target fixes its element up and
    // writes the row loss
#pragma unroll
    for (int v = 0; v < VPT; v++) {
        const int c = column(v);
        if (c < classes) {
            Pack<T> g;
            const bool has_target = target >= c && target < c + N;
#pragma unroll
            for (int j = 0; j < N; j++) {
                const float xv = raw[v].get(j);
                const float e = exponential(xv);
                float gv = e * gscale;
                if (has_target && c + j == target) {
                    row_loss[row] = -logf(e * inv + 1e-8f);
                    if (target_logit_out) target_logit_out[row] = xv;
                    gv -= scale;
                }
                g.set(j, gv);
            }
            store(c, g, std::integral_constant<bool, STREAM>{});
        }
    }
    if (WANT_ARGMAX && threadIdx.x == 0 && argmax_out) argmax_out[row] = am.i;
}

// Generic row kernel for class counts that do not fit the register-resident variants and for
// unaligned buffers: three passes over the row (the 2nd and 3rd hit L2).
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void ce_generic_kernel(const T* __restrict__ logits, const int32_t* __restrict__ targets,
                                                             T* __restrict__ dlogits, float* __restrict__ row_loss,
                                                             int32_t* __restrict__ argmax_out, float* __restrict__ target_logit_out,
                                                             int classes, float scale) {
    constexpr int W = THREADS / kWave;
    __shared__ float s_f[W];
    __shared__ int s_i[W];
    const size_t row = blockIdx.x;
    const int target = targets[row];
    const T* xr = logits + row * classes;
    T* gr = dlogits + row * classes;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (target < 0 || target >= classes) {
        for (int c = threadIdx.x; c < classes; c += THREADS) gr[c] = from_f32<T>(0.f);
        if (threadIdx.x == 0) {
            row_loss[row] = 0.f;
            if (argmax_out) argmax_out[row] = -1;
            if (target_logit_out) target_logit_out[row] = 0.f;
        }
        return;
    }
    ArgMax am{-INFINITY, 0x7fffffff};
    for (int c = threadIdx.x; c < classes; c += THREADS) {
        const float f = to_f32(xr[c]);
        if (f > am.v) {
            am.v = f;
            am.i = c;
        }
    }
    am = wave_argmax(am);
    if (W > 1) {
        if (lane == 0) {
            s_f[wid] = am.v;
            s_i[wid] = am.i;
        }
        __syncthreads();
        am = ArgMax{s_f[0], s_i[0]};
        for (int k = 1; k < W; k++) am = argmax_combine(am, ArgMax{s_f[k], s_i[k]});
        __syncthreads();
    }
    const float mx = am.v;
    float sum = 0.f;
    for (int c = threadIdx.x; c < classes; c += THREADS) sum += __expf(to_f32(xr[c]) - mx);
    sum = block_sum<THREADS>(sum, s_f);
    const float inv = 1.0f / sum;
    for (int c = threadIdx.x; c < classes; c += THREADS) {
        const float xv = to_f32(xr[c]);
        float p = __expf(xv - mx) * inv;
        if (c == target) {
            row_loss[row] = -logf(p + 1e-8f);
            if (target_logit_out) target_logit_out[row] = xv;
            p -= 1.0f;
        }
        gr[c] = from_f32<T>(p * scale);
    }
    if (threadIdx.x == 0 && argmax_out) argmax_out[row] = am.i;
}

// loss = normalizer * sum_rows row_loss, summed by one block in a fixed order.
__global__ __launch_bounds__(1024) void ce_loss_reduce_kernel(const float* __restrict__ row_loss, float* __restrict__ loss_out,
                                                              size_t rows, float normalizer) {
    __shared__ float s[1024 / kWave];
    float acc = 0.f;
    for (size_t r = threadIdx.x; r < rows; r += 1024) acc += row_loss[r];
    acc = block_sum<1024>(acc, s);
    if (threadIdx.x == 0) loss_out[0] = acc * normalizer;
}

template <typename T, int THREADS, int VPT, bool RAGGED>
void launch_fused(eisen_ctx* ctx, const void* logits, const int32_t* targets, void* dlogits, float* row_loss,
                  int32_t* argmax_out, float* target_logit_out, size_t rows, size_t classes, float scale) {
    if (argmax_out)
        ce_fused_kernel<T, THREADS, VPT, true, RAGGED><<<dim3((unsigned)rows), dim3(THREADS), 0, ctx->stream>>>(
            (const T*)logits, targets, (T*)dlogits, row_loss, argmax_out, target_logit_out, (int)rows, (int)classes, scale);
    else
        ce_fused_kernel<T, THREADS, VPT, false, RAGGED><<<dim3((unsigned)rows), dim3(THREADS), 0, ctx->stream>>>(
            (const T*)logits, targets, (T*)dlogits, row_loss, argmax_out, target_logit_out, (int)rows, (int)classes, scale);
}

template <typename T>
int ce_dispatch(eisen_ctx* ctx, const void* logits, const int32_t* targets, void* dlogits, float* row_loss,
                int32_t* argmax_out, float* target_logit_out, size_t rows, size_t classes, float scale) {
    constexpr int N = Pack<T>::N;
    const bool whole = classes % N == 0;
    const size_t packets = whole ? classes / N : (classes + 2 * N - 2) / N;  // that a row may touch
#define CE_ARGS ctx, logits, targets, dlogits, row_loss, argmax_out, target_logit_out, rows, classes, scale
#define CE_FUSED(THREADS, VPT) do { if (whole) launch_fused<T, THREADS, VPT, false>(CE_ARGS); else launch_fused<T, THREADS, VPT, true>(CE_ARGS); } while (0)
    // one wave per row up to 256 packets (no barriers, and a row of 38 packets does not hold four waves): 16000 rows of 301 bf16
    // 17.1 us, 25.6 with 256 threads; 16000 x 1000 28.3 -> 19.8
    const bool aligned = eisen_aligned(logits, 16) && eisen_aligned(dlogits, 16);
    if (aligned && packets <= 64 * 1) CE_FUSED(64, 1);
    else if (aligned && packets <= 64 * 2) CE_FUSED(64, 2);
    else if (aligned && packets <= 64 * 4) CE_FUSED(64, 4);
    else if (aligned && packets <= 256 * 2) CE_FUSED(256, 2);
    else if (aligned && packets <= 256 * 4) CE_FUSED(256, 4);
    else if (aligned && packets <= 512 * 4) CE_FUSED(512, 4);
    else if (aligned && packets <= 512 * 8) CE_FUSED(512, 8);
    else if (aligned && packets <= 1024 * 8) CE_FUSED(1024, 8);
    else if (aligned && packets <= 1024 * 16) CE_FUSED(1024, 16);
    else
        ce_generic_kernel<T, 512><<<dim3((unsigned)rows), dim3(512), 0, ctx->stream>>>(
            (const T*)logits, targets, (T*)dlogits, row_loss, argmax_out, target_logit_out, (int)classes, scale);
#undef CE_FUSED
#undef CE_ARGS
    EISEN_LAUNCH_CHECK(ctx, "ce kernel");
    return 0;
}

}  // namespace

extern "C" int eisen_hip_cross_entropy(eisen_ctx* ctx, const void* logits, const int32_t* targets, void* dlogits,
                                       float* row_loss, float* loss_out, int32_t* argmax_out, float* target_logit_out,
                                       int dtype, size_t rows, size_t classes, float normalizer, float grad_scale) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, logits && targets && dlogits && row_loss && loss_out, EISEN_E_ARG, "cross_entropy: null pointer");
    EISEN_REQUIRE(ctx, eisen_dtype_ok(dtype), EISEN_E_ARG, "cross_entropy: unknown dtype %d", dtype);
    EISEN_REQUIRE(ctx, rows > 0 && rows < (size_t(1) << 31), EISEN_E_SHAPE, "cross_entropy: rows %zu out of range", rows);
    EISEN_REQUIRE(ctx, classes > 0 && classes < (size_t(1) << 30), EISEN_E_SHAPE, "cross_entropy: classes %zu out of range", classes);
    const float scale = normalizer * grad_scale;
    // algorithmic bytes: logits read once, dlogits written once, targets read, row losses written
    EisenProfScope prof(ctx, dtype == EISEN_BF16 ? "ce_fused_bf16" : "ce_fused_f32",
                        2.0 * (double)rows * (double)classes * (double)eisen_dtype_size(dtype) + 8.0 * (double)rows);
    int rc = dtype == EISEN_F32
                 ? ce_dispatch<float>(ctx, logits, targets, dlogits, row_loss, argmax_out, target_logit_out, rows, classes, scale)
                 : ce_dispatch<bf16_t>(ctx, logits, targets, dlogits, row_loss, argmax_out, target_logit_out, rows, classes, scale);
    if (rc) return rc;
    ce_loss_reduce_kernel<<<1, 1024, 0, ctx->stream>>>(row_loss, loss_out, rows, normalizer);
    EISEN_LAUNCH_CHECK(ctx, "ce_loss_reduce_kernel");
    return 0;
}

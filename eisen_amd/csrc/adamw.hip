// Fused multi-tensor AdamW over f32 master weights, global gradient norm, zero_grad.
// One launch covers every parameter tensor: a table of slots with each tensor's first workgroup maps a workgroup to its tensor; up to 64 of them
// travel with the launch, more stand in device memory.  HBM-bound: 16 B read each of
// w, g, m, v and 16 B written each of w, m, v per packet (+ 8 B for the bf16 copy).
#include "device_utils.cuh"
#include "runtime.h"

namespace {

constexpr int kThreads = 256;
constexpr int kChunk = kThreads * 4 * 4;  // elements per workgroup: 4 float4 packets per thread

struct SlotDev {
    float* w;
    const float* g;
    float* m;
    float* v;
    bf16_t* wb;
    unsigned long long n;
};
// The table of a launch.  Up to kInline slots are part of its arguments: a copy to the device is a launch of its own in front of a kernel that takes a few
// microseconds for a small model (gradient norm and update, two copies: the step of the smallest model 303 -> 280 us, 150 M parameters in 40 tensors 937 -> 918).
constexpr int kInline = 64;
struct SlotsInline {
    int n_slots;
    unsigned first_block[kInline];  // index of a tensor's first workgroup
    SlotDev slot[kInline];
};
struct SlotsDevice {
    int n_slots;
    const unsigned* first_block;
    const SlotDev* slot;
};
__device__ __forceinline__ int find_slot(const SlotsInline& t, unsigned block) {  // every lane looks at one
    const int lane = threadIdx.x & 63;
    return __popcll(__ballot(lane < t.n_slots && t.first_block[lane] <= block)) - 1;
}
__device__ __forceinline__ int find_slot(const SlotsDevice& t, unsigned block) {
    int lo = 0, hi = t.n_slots - 1;  // last slot with first_block <= block
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (t.first_block[mid] <= block) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));
// streaming access: optimizer state is touched once per step and never reused from cache
__device__ __forceinline__ float4 nt_load4(const float* p) {
    const f32x4_t t = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p));
    return make_float4(t[0], t[1], t[2], t[3]);
}
__device__ __forceinline__ void nt_store4(float* p, float4 v) {
    f32x4_t t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<f32x4_t*>(p));
}

struct AdamParams {
    float lr, beta1, beta2, eps, wd, bc1, bc2;
};

// src/nn/optim.rs:533-542: decayed = w(1 - lr*wd); m = b1 m + (1-b1) g; v = b2 v + (1-b2) g g;
// w = decayed - lr*(m*bc1)/(sqrt(v*bc2) + eps)
__device__ __forceinline__ void adam_elem(float& w, float g, float& m, float& v, const AdamParams& p) {
    const float decayed = w * (1.0f - p.lr * p.wd);
    m = p.beta1 * m + (1.0f - p.beta1) * g;
    v = p.beta2 * v + (1.0f - p.beta2) * g * g;
    const float m_hat = m * p.bc1;
    const float v_hat = v * p.bc2;
    w = decayed - p.lr * m_hat / (sqrtf(v_hat) + p.eps);
}

template <class Slots>
__global__ __launch_bounds__(kThreads) void adamw_kernel(Slots table, AdamParams p, const float* __restrict__ grad_scale) {
    const int si = __builtin_amdgcn_readfirstlane(find_slot(table, blockIdx.x));
    const SlotDev s = table.slot[si];
    const size_t base = (size_t)(blockIdx.x - table.first_block[si]) * kChunk;
    const float gs = grad_scale ? grad_scale[0] : 1.0f;
    // All 16 loads of the thread are issued before the first use: 16 KB per stream and workgroup in flight.  The last
    // s.n % 4 elements of a tensor (bases are 16-byte aligned, so only they are no whole packet) are taken by one thread each.
    // 150 M parameters in 40 tensors of any size, bf16 copies, with the gradient norm: 932 us; 1697 us with whole tensors
    // of n % 4 != 0 taken element by element.  Bound by HBM (4.8 of the 5.1 TB/s a copy reaches).
    float4 w[4], g[4], m[4], v[4];
    bool on[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const size_t e = base + ((size_t)u * kThreads + threadIdx.x) * 4;
        on[u] = e + 4 <= s.n;
        if (on[u]) {
            w[u] = nt_load4(s.w + e);
            g[u] = nt_load4(s.g + e);
            m[u] = nt_load4(s.m + e);
            v[u] = nt_load4(s.v + e);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (!on[u]) continue;
        const size_t e = base + ((size_t)u * kThreads + threadIdx.x) * 4;
        adam_elem(w[u].x, g[u].x * gs, m[u].x, v[u].x, p);
        adam_elem(w[u].y, g[u].y * gs, m[u].y, v[u].y, p);
        adam_elem(w[u].z, g[u].z * gs, m[u].z, v[u].z, p);
        adam_elem(w[u].w, g[u].w * gs, m[u].w, v[u].w, p);
        nt_store4(s.w + e, w[u]);
        nt_store4(s.m + e, m[u]);
        nt_store4(s.v + e, v[u]);
        if (s.wb) {
            bf16x4 b;
            b[0] = (bf16_t)w[u].x; b[1] = (bf16_t)w[u].y; b[2] = (bf16_t)w[u].z; b[3] = (bf16_t)w[u].w;
            *reinterpret_cast<bf16x4*>(s.wb + e) = b;
        }
    }
    const size_t whole = s.n & ~(size_t)3;
    if (whole >= base && whole < base + kChunk && threadIdx.x < s.n - whole) {
        const size_t e = whole + threadIdx.x;
        float w1 = s.w[e], m1 = s.m[e], v1 = s.v[e];
        adam_elem(w1, s.g[e] * gs, m1, v1, p);
        s.w[e] = w1; s.m[e] = m1; s.v[e] = v1;
        if (s.wb) s.wb[e] = (bf16_t)w1;
    }
}

template <class Slots>
__global__ __launch_bounds__(kThreads) void zero_grads_kernel(Slots table) {
    const int si = __builtin_amdgcn_readfirstlane(find_slot(table, blockIdx.x));
    const SlotDev s = table.slot[si];
    const size_t base = (size_t)(blockIdx.x - table.first_block[si]) * kChunk;
    float* g = const_cast<float*>(s.g);
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const size_t e = base + ((size_t)u * kThreads + threadIdx.x) * 4;
        if (e >= s.n) break;
        if (e + 4 <= s.n) *reinterpret_cast<float4*>(g + e) = make_float4(0.f, 0.f, 0.f, 0.f);
        else
            for (size_t j = e; j < s.n; j++) g[j] = 0.f;
    }
}

// stage 1: one f64 partial per workgroup (src/nn/optim.rs:258-262 accumulates x*x in f64)
template <class Slots>
__global__ __launch_bounds__(kThreads) void sumsq_kernel(Slots table, double* __restrict__ partial) {
    __shared__ double sh[kThreads / kWave];
    const int si = __builtin_amdgcn_readfirstlane(find_slot(table, blockIdx.x));
    const SlotDev s = table.slot[si];
    const size_t base = (size_t)(blockIdx.x - table.first_block[si]) * kChunk;
    double acc = 0.0;
    float4 g[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const size_t e = base + ((size_t)u * kThreads + threadIdx.x) * 4;
        g[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e + 4 <= s.n) {
            g[u] = *reinterpret_cast<const float4*>(s.g + e);
        } else if (e < s.n) {  // the tensor's last, partial packet: the elements it lacks add nothing
            g[u].x = s.g[e];
            if (e + 1 < s.n) g[u].y = s.g[e + 1];
            if (e + 2 < s.n) g[u].z = s.g[e + 2];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        acc += (double)g[u].x * (double)g[u].x;
        acc += (double)g[u].y * (double)g[u].y;
        acc += (double)g[u].z * (double)g[u].z;
        acc += (double)g[u].w * (double)g[u].w;
    }
    acc = wave_sum_f64(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kThreads / kWave; k++) t += sh[k];
        partial[blockIdx.x] = t;
    }
}
// (The workgroup that arrives last adding the partials up itself costs 23 ns per workgroup, more than a launch from 200 on.)
// stage 2: one workgroup, fixed order; writes norm and clip coefficient (src/nn/optim.rs:282-287)
__global__ __launch_bounds__(1024) void norm_finish_kernel(const double* __restrict__ partial, size_t n, float max_norm, float* __restrict__ out) {
    __shared__ double sh[1024 / kWave];
    double acc = 0.0;
    for (size_t i = threadIdx.x; i < n; i += 1024) acc += partial[i];
    acc = wave_sum_f64(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < 1024 / kWave; k++) t += sh[k];
        const float norm = (float)sqrt(t);
        float coef = 1.0f;
        if (norm > 0.0f) coef = fminf(max_norm / (norm + 1e-6f), 1.0f);
        out[0] = norm;
        out[1] = coef;
    }
}

// Checks the slots, forms the launch's table and calls launch(table, workgroups).
template <class F>
int with_slots(eisen_ctx* ctx, const eisen_param_slot* slots, size_t n_slots, bool need_moments, const char* who, F&& launch) {
    EISEN_REQUIRE(ctx, slots && n_slots > 0 && n_slots < (size_t(1) << 20), EISEN_E_ARG, "%s: bad slot table", who);
    SlotsInline small;
    std::vector<char> large;  // [slots | first workgroups]
    if (n_slots > (size_t)kInline) large.resize(n_slots * (sizeof(SlotDev) + sizeof(unsigned)));
    SlotDev* slot = large.empty() ? small.slot : reinterpret_cast<SlotDev*>(large.data());
    unsigned* first = large.empty() ? small.first_block : reinterpret_cast<unsigned*>(large.data() + n_slots * sizeof(SlotDev));
    size_t blocks = 0;
    for (size_t i = 0; i < n_slots; i++) {
        const eisen_param_slot& s = slots[i];
        EISEN_REQUIRE(ctx, s.g && s.n > 0, EISEN_E_ARG, "%s: slot %zu has a null gradient or zero size", who, i);
        EISEN_REQUIRE(ctx, !need_moments || (s.w && s.m && s.v), EISEN_E_ARG, "%s: slot %zu lacks w/m/v", who, i);
        EISEN_REQUIRE(ctx, eisen_aligned(s.g, 16) && eisen_aligned(s.w, 16) && eisen_aligned(s.m, 16) && eisen_aligned(s.v, 16) && eisen_aligned(s.w_bf16, 8),
                      EISEN_E_ALIGN, "%s: slot %zu buffers must be 16-byte aligned", who, i);
        EISEN_REQUIRE(ctx, blocks < (size_t(1) << 31), EISEN_E_SHAPE, "%s: too many elements for one launch", who);
        slot[i] = SlotDev{s.w, s.g, s.m, s.v, (bf16_t*)s.w_bf16, (unsigned long long)s.n};
        first[i] = (unsigned)blocks;
        blocks += eisen_ceil_div(s.n, kChunk);
    }
    EISEN_REQUIRE(ctx, blocks < (size_t(1) << 31), EISEN_E_SHAPE, "%s: too many elements for one launch", who);
    if (large.empty()) {
        small.n_slots = (int)n_slots;
        return launch(small, (unsigned)blocks);
    }
    void* dev = nullptr;
    int rc = eisen_hip_malloc(ctx, large.size(), &dev);
    if (rc) return rc;
    rc = eisen_hip_htod(ctx, dev, large.data(), large.size());
    if (!rc) rc = launch(SlotsDevice{(int)n_slots, reinterpret_cast<const unsigned*>(static_cast<char*>(dev) + n_slots * sizeof(SlotDev)), static_cast<const SlotDev*>(dev)}, (unsigned)blocks);
    const int rc_free = eisen_hip_free(ctx, dev);
    return rc ? rc : rc_free;
}

}  // namespace

extern "C" int eisen_hip_adamw_step(eisen_ctx* ctx, const eisen_param_slot* slots, size_t n_slots, float lr, float beta1,
                                    float beta2, float eps, float weight_decay, float bc1, float bc2,
                                    const float* grad_scale_device) {
    EISEN_CHECK_CTX(ctx);
    return with_slots(ctx, slots, n_slots, true, "adamw_step", [&](const auto& table, unsigned blocks) -> int {
        AdamParams p{lr, beta1, beta2, eps, weight_decay, bc1, bc2};
        double bytes = 0.0;  // per parameter: w, g, m, v read, w, m, v written (28 B) and the bf16 copy written where there is one
        for (size_t i = 0; i < n_slots; i++) bytes += (double)slots[i].n * (slots[i].w_bf16 ? 30.0 : 28.0);
        EisenProfScope prof(ctx, "adamw", bytes);
        adamw_kernel<<<blocks, kThreads, 0, ctx->stream>>>(table, p, grad_scale_device);
        EISEN_LAUNCH_CHECK(ctx, "adamw_kernel");
        return 0;
    });
}

extern "C" int eisen_hip_zero_grads(eisen_ctx* ctx, const eisen_param_slot* slots, size_t n_slots) {
    EISEN_CHECK_CTX(ctx);
    return with_slots(ctx, slots, n_slots, false, "zero_grads", [&](const auto& table, unsigned blocks) -> int {
        zero_grads_kernel<<<blocks, kThreads, 0, ctx->stream>>>(table);
        EISEN_LAUNCH_CHECK(ctx, "zero_grads_kernel");
        return 0;
    });
}

extern "C" int eisen_hip_grad_norm(eisen_ctx* ctx, const eisen_param_slot* slots, size_t n_slots, float max_norm,
                                   float* out_device) {
    EISEN_CHECK_CTX(ctx);
    EISEN_REQUIRE(ctx, out_device != nullptr, EISEN_E_ARG, "grad_norm: null output");
    return with_slots(ctx, slots, n_slots, false, "grad_norm", [&](const auto& table, unsigned blocks) -> int {
        void* ws = nullptr;
        int rc = eisen_workspace(ctx, blocks * sizeof(double), &ws);
        if (rc) return rc;
        double bytes = 0.0;
        for (size_t i = 0; i < n_slots; i++) bytes += (double)slots[i].n * 4.0;
        EisenProfScope prof(ctx, "grad_sumsq", bytes);
        sumsq_kernel<<<blocks, kThreads, 0, ctx->stream>>>(table, (double*)ws);
        EISEN_LAUNCH_CHECK(ctx, "sumsq_kernel");
        norm_finish_kernel<<<1, 1024, 0, ctx->stream>>>((const double*)ws, blocks, max_norm, out_device);
        EISEN_LAUNCH_CHECK(ctx, "norm_finish_kernel");
        return 0;
    });
}

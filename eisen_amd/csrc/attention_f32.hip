// f32 attention on the matrix cores (head_dim up to 128), forward and backward; see attention.hip for the formulas and the
// reference lines.  Instantiated per head_dim rounded up to a class of 8 * K8.
//
// v_mfma_f32_32x32x2_f32 takes 64 cycles for 32 x 32 x 2 products, so a wave reads about 16 bytes of operands per cycle and CU
// whatever it does: the caches deliver that, and every operand goes from memory straight to the registers of the wave that
// multiplies it.  No LDS tiles and no barrier in the loops; the loads of the next tile's rows are issued before the products
// that hide them.  What bounds the kernels is the length of a wave's chain of MFMAs times how many of the 1024 SIMDs have one:
// the keys (forward, dQ) or the (query head, query tile) items (dK/dV) of a workgroup are dealt to as many waves as the grid
// lacks, and their partial results meet in LDS once at the end.
//
// Layouts.  A contraction over head_dim takes four consecutive d per lane (8 kk + 4 (lane / 32) + 0..3) from both operands.
// Scores come out transposed for the query-stationary kernels (S^T = K Q^T: a lane owns query lane % 32 and keys acc_row(v, h))
// and as S for the key-stationary one (a lane owns a key), which is the order in which register v is an operand of step v of
// the second product.  The results are O^T, dQ^T, dK^T, dV^T: a lane holds four consecutive d of one row, as the stores (and
// the rotary backward's pairs) want them.
#include <cmath>

#include "attention_common.cuh"
#include "attention_f32_plan.h"

namespace {

struct __attribute__((packed, aligned(4))) Quad { float v[4]; };

// Rows `stride` apart.  A load takes the tile's origin in scalar registers and an unsigned 32-bit byte offset per
// lane, so that the loops spend few vector instructions on addresses (64-bit sums per lane and load had been a third of those of a
// dK/dV item).  A negative stride moves the origin to the lowest of 32 rows.  FAR: |stride| >= 2^24, which 32 rows of such an offset
// do not reach; 64-bit sums, in kernels of their own (128 positions 2^24 apart, 8 heads of 128, forward and backward in us: 14 and 47; on the
// plain kernels 237 and 979).
template <bool FAR>
struct RowStride {
    long long stride;
    int low;  // elements
    __device__ __forceinline__ explicit RowStride(long long s) : stride(s), low(FAR ? 0 : min(0, 31 * (int)s)) {}
};
template <class T>
__device__ __forceinline__ const T& at_bytes(const float* origin, unsigned bytes) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(origin) + bytes);
}
// This lane's share of row first_row + c (the last row, past the end): d = 8 kk + 4 h + 0..3.  FULL: head_dim is 8 * K8.  Where it is
// not, a load may stand behind a branch of its lanes, and the row's own address in two registers does better than an offset that every
// branch adds up again (offset / address, us: 8 x 512, 8 heads of 100 forward 88 / 77, backward 395 / 319; 1 x 800, 8 of 100 64 / 54 and
// 159 / 133; 16 x 512, 8 of 40 backward 264 / 243; 16 x 512, 8 of 20 157 / 135).
template <int K8, bool FULL, bool FAR>
__device__ __forceinline__ void load_row(const float* base, const RowStride<FAR>& rs, int first_row, int rows, int hd, int c, int h, float (&f)[K8][4]) {
    if (FULL && !FAR) {
        const float* origin = base + first_row * rs.stride + rs.low;
        const unsigned off = (unsigned)(min(c, rows - 1 - first_row) * (int)rs.stride - rs.low) * 4u + 16u * h;
#pragma unroll
        for (int kk = 0; kk < K8; kk++) {
            const Quad q = at_bytes<Quad>(origin + 8 * kk, off);
#pragma unroll
            for (int j = 0; j < 4; j++) f[kk][j] = q.v[j];
        }
    } else {
        const float* row = base + (long long)min(first_row + c, rows - 1) * rs.stride;
#pragma unroll
        for (int kk = 0; kk < K8; kk++) {
            const int d = 8 * kk + 4 * h;
            if (FULL || d + 4 <= hd) {
                const Quad q = *reinterpret_cast<const Quad*>(row + d);
#pragma unroll
                for (int j = 0; j < 4; j++) f[kk][j] = q.v[j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) f[kk][j] = d + j < hd ? row[d + j] : 0.f;
            }
        }
    }
}
// Columns d = 32 dt + lane % 32 of the 32 rows at first_row, in the order of a score tile's registers.  Rows past the end
// repeat the last one (their weight is zero).
template <int K8, bool FULL, bool FAR>
__device__ __forceinline__ void load_column(const float* base, const RowStride<FAR>& rs, int first_row, int rows, int hd, int c, int h, int dt, float (&f)[16]) {
    const float* origin = base + first_row * rs.stride + rs.low + 32 * dt;
    const int d = 32 * dt + c, last = rows - 1 - first_row, stride = (int)rs.stride;
    const bool in = FULL ? (32 * dt + 32 <= 8 * K8 || d < 8 * K8) : d < hd;
    if (FAR) {
#pragma unroll
        for (int v = 0; v < 16; v++) f[v] = in ? base[min(first_row + acc_row(v, h), rows - 1) * rs.stride + d] : 0.f;
        return;
    }
#pragma unroll
    for (int v = 0; v < 16; v++) {  // the products are scalar
        const int r0 = min(acc_row(v, 0), last) * stride, r1 = min(acc_row(v, 1), last) * stride;
        const unsigned off = (unsigned)((h ? r1 : r0) - rs.low + c) * 4u;
        f[v] = in ? at_bytes<float>(origin, off) : 0.f;
    }
}
template <int K8, int DT, bool FULL, bool FAR>
__device__ __forceinline__ void load_columns(const float* base, const RowStride<FAR>& rs, int first_row, int rows, int hd, int c, int h, float (&f)[DT][16]) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++) load_column<K8, FULL>(base, rs, first_row, rows, hd, c, h, dt, f[dt]);
}
// registers of a transposed result tile -> row `row` (d = 32 dt + 8 vg + 4 h + 0..3)
template <int K8, bool FULL>
__device__ __forceinline__ void store_quad(float* row, int d, int hd, const float (&x)[4]) {
    if (FULL ? d < 8 * K8 : d + 4 <= hd) {
        Quad q;
#pragma unroll
        for (int e = 0; e < 4; e++) q.v[e] = x[e];
        *reinterpret_cast<Quad*>(row + d) = q;
    } else if (!FULL) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (d + e < hd) row[d + e] = x[e];
    }
}
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int v = 0; v < 16; v++) z[v] = 0.f;
    return z;
}
template <int K8>
__device__ __forceinline__ f32x16 row_product(const float (&a)[K8][4], const float (&b)[K8][4], f32x16 acc) {
#pragma unroll
    for (int kk = 0; kk < K8; kk++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[kk][j], b[kk][j], acc, 0, 0, 0);
    return acc;
}

// Rows that are masked for a lane have weight zero in the second product, and zero times an Inf or NaN would still reach the
// lane's result: a query must not depend on what stands in later rows of K and V, nor a key on earlier rows of Q and dO.  The
// tiles with masked pairs are therefore looked at; if one holds a value that is not finite, such values are taken out of the
// operand, and behind the loop, where the registers are free, put_back_nonfinite() gives them to the lanes that do see their
// row.  The look is one instruction per value: of V itself in the forward pass, of the first products' 16 results in the
// backward pass (a row of Q, K or dO that is not finite makes them not finite).  16 x 83, one head of 64, forward and
// backward in three launches: 8.6 + 27.2 us without the look, 8.7 + 27.9 with it, 9.0 + 30.1 with every operand of such tiles cleaned.
__device__ __forceinline__ float look(float x, float seen) { return fmaf(x, 0.f, seen); }  // stays 0, or becomes NaN for good
__device__ __forceinline__ bool any_nan(float seen) { return __builtin_amdgcn_ballot_w64(seen != seen) != 0; }
template <int DT>
__device__ __forceinline__ bool take_out_nonfinite(float (&col)[DT][16]) {  // whether there were any, the same in all lanes
    bool found = false;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const bool finite = fabsf(col[dt][v]) < INFINITY;
            found |= !finite;
            col[dt][v] = finite ? col[dt][v] : 0.f;
        }
    return __builtin_amdgcn_ballot_w64(found) != 0;
}
// +-Inf for the weights P of V and dO, which are not negative (POSITIVE), NaN for the others and for NaN.
template <bool POSITIVE, int K8, int DT, bool FULL, bool FAR, class Visible>
__device__ __forceinline__ void put_back_nonfinite(const float* base, const RowStride<FAR>& stride, int first_row, int rows, int hd, int c, int h, f32x16 (&acc)[DT],
                                                   Visible visible) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
        float x[16];
        load_column<K8, FULL>(base, stride, first_row, rows, hd, c, h, dt, x);
#pragma unroll
        for (int sign = 0; sign < (POSITIVE ? 2 : 1); sign++) {
            f32x16 seen = zero16();  // how many such values (of this sign, or NaN) the lane's row sees in each column
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const bool bad = !(fabsf(x[v]) < INFINITY) && !(POSITIVE && (sign == 0 ? x[v] < 0.f : x[v] > 0.f));
                seen = __builtin_amdgcn_mfma_f32_32x32x2f32(bad ? 1.f : 0.f, visible(v) ? 1.f : 0.f, seen, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 16; v++) acc[dt][v] += seen[v] > 0.f ? (!POSITIVE ? NAN : sign == 0 ? INFINITY : -INFINITY) : 0.f;
        }
    }
}

// workgroup -> (query block or key block, head, batch): heads and batches fastest, the longest causal blocks first
struct RowBlock { int blk, head, b; };
__device__ __forceinline__ RowBlock decode_block(int id, int heads, int B, int n_blk, bool descending) {
    const int per = heads * B;
    const int i = id / per, r = id % per;
    return RowBlock{descending ? n_blk - 1 - i : i, r % heads, r / heads};
}

template <int K8>
constexpr int kMaxWaves = f32_attn_max_waves(K8);
extern __shared__ float meet[];  // where the waves of a workgroup meet: as much as the launch's waves need (attention_f32_plan.h)

// (up to head size 16 four waves to a SIMD: one register more than that allows made 7 x 1170, 3 heads of 8 62.5 us instead of 54.5)
template <int K8, bool FULL, bool FAR>
__global__ __launch_bounds__(64 * kMaxWaves<K8>, K8 <= 2 ? 4 : kMaxWaves<K8> / 4) void attn_f32_fwd_kernel(AttnArgs a) {
    constexpr int DT = (K8 + 3) / 4;
    const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    const RowBlock rb = decode_block(blockIdx.x, a.Hq, a.B, (a.S + 31) / 32, a.causal);
    const int q0 = rb.blk * 32, q = min(q0 + c, a.S - 1);
    const long long qoff = rb.b * a.q_sb + rb.head * a.q_sh + (long long)q * a.q_ss;
    const long long kvoff = rb.b * a.k_sb + (rb.head / a.G) * a.k_sh;
    const float* Kp = static_cast<const float*>(a.K) + kvoff;
    const float* Vp = static_cast<const float*>(a.V) + kvoff;
    const RowStride<FAR> qs(a.q_ss), ks(a.k_ss);
    float qf[K8][4], kf[K8][4];
    load_row<K8, FULL>(static_cast<const float*>(a.Q) + rb.b * a.q_sb + rb.head * a.q_sh, qs, q0, a.S, a.hd, c, h, qf);
    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = zero16();
    float m = -INFINITY, l = 0.f;  // m in units of log2
    int odd_at = -1;               // first row of the tile with masked pairs, if it holds a value that is not finite
    const int n_kt = a.causal ? min(rb.blk + 1, (a.S + 31) / 32) : (a.S + 31) / 32;
    if (wave < n_kt) load_row<K8, FULL>(Kp, ks, wave * 32, a.S, a.hd, c, h, kf);
    for (int kt = wave; kt < n_kt; kt += nw) {
        float vc[DT][16];
        load_columns<K8, DT, FULL>(Vp, ks, kt * 32, a.S, a.hd, c, h, vc);
        f32x16 s = row_product<K8>(kf, qf, zero16());
        if (kt + nw < n_kt) load_row<K8, FULL>(Kp, ks, (kt + nw) * 32, a.S, a.hd, c, h, kf);
        const int k0 = kt * 32, lim = (a.causal ? q : a.S - 1) - k0;  // tile rows above lim are masked
        if (k0 + 32 > a.S || (a.causal && k0 + 31 > q0)) {
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (acc_row(v, h) > lim) s[v] = -INFINITY;
            float seen = 0.f;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) seen = look(vc[dt][v], seen);
            if (any_nan(seen)) {
                take_out_nonfinite(vc);
                odd_at = k0;
            }
        }
        float mx = s[0];
#pragma unroll
        for (int v = 1; v < 16; v++) mx = fmaxf(mx, s[v]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * a.scale_log2e;
        if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
            const float mn = fmaxf(m, mx), alpha = m == -INFINITY ? 0.f : fast_exp2(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) o[dt][v] *= alpha;
        }
        const float mu = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            s[v] = fast_exp2(fmaf(s[v], a.scale_log2e, -mu));
            l += s[v];
        }
#pragma unroll
        for (int v = 0; v < 16; v++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vc[dt][v], s[v], o[dt], 0, 0, 0);
    }
    if (odd_at >= 0) {
        const int lim = (a.causal ? q : a.S - 1) - odd_at;
        put_back_nonfinite<true, K8, DT, FULL>(Vp, ks, odd_at, a.S, a.hd, c, h, o, [&](int v) { return acc_row(v, h) <= lim; });
    }
    l += __shfl_xor(l, 32, 64);
    if (nw > 1) {  // the waves' keys are disjoint: (m, l, O) of each, added in wave order against the common maximum
        auto share = [&](int w) { return meet + f32_attn_fwd_meet(DT, w); };  // of wave w > 0
        if (wave > 0) {
            float* p = share(wave);
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) p[(dt * 16 + v) * 64 + lane] = o[dt][v];
            p[DT * 16 * 64 + lane] = m;
            p[DT * 16 * 64 + 64 + lane] = l;
        }
        __syncthreads();
        if (wave > 0) return;
        float mn = m;
        for (int w = 1; w < nw; w++) mn = fmaxf(mn, share(w)[DT * 16 * 64 + lane]);
        const float a0 = m == -INFINITY ? 0.f : fast_exp2(m - mn);
        l *= a0;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) o[dt][v] *= a0;
        for (int w = 1; w < nw; w++) {
            const float* p = share(w);
            const float mw = p[DT * 16 * 64 + lane], aw = mw == -INFINITY ? 0.f : fast_exp2(mw - mn);
            l += p[DT * 16 * 64 + 64 + lane] * aw;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) o[dt][v] += p[(dt * 16 + v) * 64 + lane] * aw;
        }
        m = mn;
    }
    if (q0 + c >= a.S) return;
    const float inv = 1.0f / l;
    float* Op = static_cast<float*>(a.Out) + qoff;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int vg = 0; vg < 4; vg++) {
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = o[dt][vg * 4 + e] * inv;
            store_quad<K8, FULL>(Op, 32 * dt + 8 * vg + 4 * h, a.hd, x);
        }
    if (h == 0) a.LSE[((long long)rb.b * a.Hq + rb.head) * a.S + q] = (m + log2f(l)) * kLn2;
}

// D = rowsum(dO o O) of this lane's row, from its two lanes' shares
template <int K8>
__device__ __forceinline__ float row_dot(const float (&x)[K8][4], const float (&y)[K8][4]) {
    float d = 0.f;
#pragma unroll
    for (int kk = 0; kk < K8; kk++)
#pragma unroll
        for (int j = 0; j < 4; j++) d += x[kk][j] * y[kk][j];
    return d + __shfl_xor(d, 32, 64);
}

// dQ^T = scale K^T dS^T of query block `id` (none, past the last: the wave only meets the others at the barrier), by nw waves of
// which this is the `wave`-th; WRITE_D: also leaves D = rowsum(dO o O) for a dK/dV launch that follows.
template <int K8, bool FULL, bool FAR, bool WRITE_D>
__device__ __forceinline__ void bwd_dq(const AttnArgs& a, int id, int wave, int nw, float* share) {
    constexpr int DT = (K8 + 3) / 4;
    const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
    const int n_t = (a.S + 31) / 32;
    const bool exists = id < n_t * a.Hq * a.B;
    const RowBlock rb = decode_block(exists ? id : 0, a.Hq, a.B, n_t, a.causal);
    const int q0 = rb.blk * 32, q = min(q0 + c, a.S - 1);
    const long long qoff = rb.b * a.q_sb + rb.head * a.q_sh;
    const long long kvoff = rb.b * a.k_sb + (rb.head / a.G) * a.k_sh;
    const long long stat = ((long long)rb.b * a.Hq + rb.head) * a.S + q;
    const float* Kp = static_cast<const float*>(a.K) + kvoff;
    const float* Vp = static_cast<const float*>(a.V) + kvoff;
    const RowStride<FAR> qs(a.q_ss), ks(a.k_ss);
    float qf[K8][4], dof[K8][4], kf[K8][4], vf[K8][4];
    load_row<K8, FULL>(static_cast<const float*>(a.dO) + qoff, qs, q0, a.S, a.hd, c, h, dof);
    load_row<K8, FULL>(static_cast<const float*>(a.O) + qoff, qs, q0, a.S, a.hd, c, h, qf);
    const float Dq = row_dot<K8>(dof, qf);
    load_row<K8, FULL>(static_cast<const float*>(a.Q) + qoff, qs, q0, a.S, a.hd, c, h, qf);
    const float lse2 = a.LSE[stat] * kLog2e;
    if (WRITE_D && exists && wave == 0 && h == 0 && q0 + c < a.S) a.D[stat] = Dq;
    f32x16 dq[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) dq[dt] = zero16();
    int odd_at = -1;  // see the forward kernel
    const int n_kt = !exists ? 0 : a.causal ? min(rb.blk + 1, n_t) : n_t;
    auto fetch = [&](int kt) {
        load_row<K8, FULL>(Kp, ks, kt * 32, a.S, a.hd, c, h, kf);
        load_row<K8, FULL>(Vp, ks, kt * 32, a.S, a.hd, c, h, vf);
    };
    if (wave < n_kt) fetch(wave);
    for (int kt = wave; kt < n_kt; kt += nw) {
        float kc[DT][16];
        load_columns<K8, DT, FULL>(Kp, ks, kt * 32, a.S, a.hd, c, h, kc);
        f32x16 s = row_product<K8>(kf, qf, zero16());
        const f32x16 dp = row_product<K8>(vf, dof, zero16());
        if (kt + nw < n_kt) fetch(kt + nw);
        const int k0 = kt * 32, lim = (a.causal ? q : a.S - 1) - k0;
        const bool masked = k0 + 32 > a.S || (a.causal && k0 + 31 > q0);
        if (masked) {
            float seen = 0.f;
#pragma unroll
            for (int v = 0; v < 16; v++) seen = look(s[v], seen);
            if (any_nan(seen)) {
                take_out_nonfinite(kc);
                odd_at = k0;
            }
        }
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = fast_exp2(fmaf(s[v], a.scale_log2e, -lse2)) * (dp[v] - Dq) * a.scale;
        if (masked) {
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (acc_row(v, h) > lim) s[v] = 0.f;
        }
#pragma unroll
        for (int v = 0; v < 16; v++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) dq[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kc[dt][v], s[v], dq[dt], 0, 0, 0);
    }
    if (odd_at >= 0) {
        const int lim = (a.causal ? q : a.S - 1) - odd_at;
        put_back_nonfinite<false, K8, DT, FULL>(Kp, ks, odd_at, a.S, a.hd, c, h, dq, [&](int v) { return acc_row(v, h) <= lim; });
    }
    if (nw > 1) {
        if (wave > 0) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) share[(((wave - 1) * DT + dt) * 16 + v) * 64 + lane] = dq[dt][v];
        }
        __syncthreads();
        if (wave > 0) return;
        for (int w = 0; w < nw - 1; w++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) dq[dt][v] += share[((w * DT + dt) * 16 + v) * 64 + lane];
    }
    if (!exists || q0 + c >= a.S) return;
    float* dQp = static_cast<float*>(a.dQ) + qoff + (long long)q * a.q_ss;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int vg = 0; vg < 4; vg++) {
            const int d = 32 * dt + 8 * vg + 4 * h;
            if (d >= (FULL ? 8 * K8 : a.hd)) continue;
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = dq[dt][vg * 4 + e];
            if (a.rope) {  // (head_dim is even; a pair beyond it is not stored)
                unrotate_pairs<1>(x, a.rope + (size_t)q * (a.hd / 2) + d / 2);
                if (d + 2 < a.hd) unrotate_pairs<1>(x + 2, a.rope + (size_t)q * (a.hd / 2) + d / 2 + 1);
            }
            store_quad<K8, FULL>(dQp, d, a.hd, x);
        }
}

// dK^T = scale Q^T dS, dV^T = dO^T P of key block `id`, summed over the query heads of the group (ascending within a wave, then
// over the waves).  OWN_D: D is formed from the rows of O here, as the dQ pass forms it, and not read.  The rows and statistics
// of an item are requested under the products of the one before, its columns under its own first products: a lane loads the
// statistics of the row it holds, and the lanes that need them ask it.
template <int K8, bool FULL, bool FAR, bool OWN_D>
__device__ __forceinline__ void bwd_dkv(const AttnArgs& a, int id, int wave, int nw) {
    constexpr int DT = (K8 + 3) / 4;
    constexpr bool AHEAD = K8 <= 8;  // (above, the registers are all taken)
    const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
    const int n_t = (a.S + 31) / 32;
    const RowBlock rb = decode_block(id, a.Hkv, a.B, n_t, false);  // ascending: the first keys see the most queries
    const int k0 = rb.blk * 32, key = min(k0 + c, a.S - 1);
    const long long kvoff = rb.b * a.k_sb + rb.head * a.k_sh;
    const RowStride<FAR> qs(a.q_ss), ks(a.k_ss);
    float kf[K8][4], vf[K8][4];
    load_row<K8, FULL>(static_cast<const float*>(a.K) + kvoff, ks, k0, a.S, a.hd, c, h, kf);
    load_row<K8, FULL>(static_cast<const float*>(a.V) + kvoff, ks, k0, a.S, a.hd, c, h, vf);
    f32x16 dk[DT], dv[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) dk[dt] = dv[dt] = zero16();
    const int qt_start = a.causal ? rb.blk : 0, per_head = n_t - qt_start, n_items = a.G * per_head;
    auto masked_tile = [&](int q0) { return (a.causal && q0 < k0 + 31) || q0 + 32 > a.S; };
    auto visible = [&](int q0, int v) {
        const int r = q0 + acc_row(v, h);
        return r < a.S && !(a.causal && k0 + c > r);
    };
    float qr[K8][4], dor[K8][4], orow[K8][4], lse_row = 0.f, d_row = 0.f;
    auto fetch = [&](int item) {
        const int hq = rb.head * a.G + item / per_head, q0 = (qt_start + item % per_head) * 32;
        const long long base = rb.b * a.q_sb + hq * a.q_sh, stat = ((long long)rb.b * a.Hq + hq) * a.S + q0;
        load_row<K8, FULL>(static_cast<const float*>(a.dO) + base, qs, q0, a.S, a.hd, c, h, dor);
        if (OWN_D) load_row<K8, FULL>(static_cast<const float*>(a.O) + base, qs, q0, a.S, a.hd, c, h, orow);
        if (OWN_D && !AHEAD) {
            d_row = row_dot<K8>(dor, orow);
            asm volatile("" : "+v"(d_row)::"memory");  // the rows of O are done with before the other operands arrive
        }
        load_row<K8, FULL>(static_cast<const float*>(a.Q) + base, qs, q0, a.S, a.hd, c, h, qr);
        const int r = min(c, a.S - 1 - q0);
        lse_row = a.LSE[stat + r];
        if (!OWN_D) d_row = a.D[stat + r];
    };
    bool odd = false;
    if (AHEAD && wave < n_items) fetch(wave);
    for (int item = wave; item < n_items; item += nw) {
        const int hq = rb.head * a.G + item / per_head, q0 = (qt_start + item % per_head) * 32;
        const long long base = rb.b * a.q_sb + hq * a.q_sh;
        if (!AHEAD) fetch(item);
        float qc[DT][16], doc[DT][16];
        auto columns_of_do = [&] { load_columns<K8, DT, FULL>(static_cast<const float*>(a.dO) + base, qs, q0, a.S, a.hd, c, h, doc); };
        auto columns_of_q = [&] { load_columns<K8, DT, FULL>(static_cast<const float*>(a.Q) + base, qs, q0, a.S, a.hd, c, h, qc); };
        columns_of_do();
        if (AHEAD) columns_of_q();
        f32x16 s = row_product<K8>(qr, kf, zero16());
        if (!AHEAD) {  // the columns of Q take the registers of its rows, which the products above have read
            asm volatile("" : "+v"(s)::"memory");
            columns_of_q();
        }
        f32x16 dp = row_product<K8>(dor, vf, zero16());
        const bool in = q0 + c < a.S;  // a query past the end has no weight
        const float d_here = OWN_D && AHEAD ? row_dot<K8>(dor, orow) : d_row, l_here = lse_row * kLog2e;
        const float l_own = in ? l_here : INFINITY, d_own = in ? d_here : 0.f;
        auto lse2 = [&](int v) { return __shfl(l_own, acc_row(v, h), 64); };
        auto D = [&](int v) { return __shfl(d_own, acc_row(v, h), 64); };
        if (AHEAD && item + nw < n_items) fetch(item + nw);
        // Up to head size 96 the tile is looked at before its operands are touched; above, where the look's registers would go to
        // scratch (1 x 800, 8 heads of 128: backward 411 -> 421 us), every such tile is cleaned.
        constexpr bool kLook = K8 <= 12;
        bool odd_here = false;
        if (kLook && masked_tile(q0)) {
            float seen = 0.f;
#pragma unroll
            for (int v = 0; v < 16; v++) seen = look(dp[v] - D(v), look(s[v], seen));
            odd_here = any_nan(seen);
        }
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = fast_exp2(fmaf(s[v], a.scale_log2e, -lse2(v)));
        if (kLook && a.causal && q0 < k0 + 31) {
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (k0 + c > q0 + acc_row(v, h)) s[v] = 0.f;
        }
#pragma unroll
        for (int v = 0; v < 16; v++) dp[v] = s[v] * (dp[v] - D(v)) * a.scale;
        if (kLook ? odd_here : masked_tile(q0)) {
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (!visible(q0, v)) s[v] = dp[v] = 0.f;  // (dp too: D of a masked query may be NaN)
            const bool odd_do = take_out_nonfinite(doc), odd_q = take_out_nonfinite(qc);
            odd |= odd_do || odd_q;
        }
#pragma unroll
        for (int v = 0; v < 16; v++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                dv[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(doc[dt][v], s[v], dv[dt], 0, 0, 0);
                dk[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(qc[dt][v], dp[v], dk[dt], 0, 0, 0);
            }
    }
    if (odd) {
        for (int item = wave; item < n_items; item += nw) {
            const int hq = rb.head * a.G + item / per_head, q0 = (qt_start + item % per_head) * 32;
            const long long base = rb.b * a.q_sb + hq * a.q_sh;
            if (!masked_tile(q0)) continue;
            put_back_nonfinite<true, K8, DT, FULL>(static_cast<const float*>(a.dO) + base, qs, q0, a.S, a.hd, c, h, dv, [&](int v) { return visible(q0, v); });
            put_back_nonfinite<false, K8, DT, FULL>(static_cast<const float*>(a.Q) + base, qs, q0, a.S, a.hd, c, h, dk, [&](int v) { return visible(q0, v); });
        }
    }
    const long long koff = kvoff + (long long)key * a.k_ss;
    float* outs[2] = {static_cast<float*>(a.dK) + koff, static_cast<float*>(a.dV) + koff};
#pragma unroll
    for (int i = 0; i < 2 * DT; i++) {  // one 32-column tile of dK or dV at a time; the waves take turns in adding up
        const int dt = i >> 1;
        f32x16 r = (i & 1) ? dv[dt] : dk[dt];
        if (nw > 1) {
            float* p = meet + (i & 1) * nw * kF32AttnTile;
#pragma unroll
            for (int v = 0; v < 16; v++) p[(wave * 16 + v) * 64 + lane] = r[v];
            __syncthreads();  // (the buffer of tile i was last read before the barrier of tile i - 1)
            if (i % nw != wave) continue;
            r = zero16();
            for (int w = 0; w < nw; w++)
#pragma unroll
                for (int v = 0; v < 16; v++) r[v] += p[(w * 16 + v) * 64 + lane];
        }
        if (k0 + c >= a.S) continue;
#pragma unroll
        for (int vg = 0; vg < 4; vg++) {
            const int d = 32 * dt + 8 * vg + 4 * h;
            if (d >= (FULL ? 8 * K8 : a.hd)) continue;
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = r[vg * 4 + e];
            if (!(i & 1) && a.rope) {
                unrotate_pairs<1>(x, a.rope + (size_t)key * (a.hd / 2) + d / 2);
                if (d + 2 < a.hd) unrotate_pairs<1>(x + 2, a.rope + (size_t)key * (a.hd / 2) + d / 2 + 1);
            }
            store_quad<K8, FULL>(outs[i & 1], d, a.hd, x);
        }
    }
}

// Both passes in one launch: the first kblocks workgroups form dK and dV of a key block each, the others dQ of as many query blocks
// as they have wq waves for.  The two do not wait for one another (the dK/dV pass forms D itself), so a grid that does not fill the
// chip takes the time of the longer pass, and in one that does either pass fills the gaps of the other (where that is not enough: F32AttnPlan).  Two launches with
// an address of its own per load, and a dK/dV item's rows requested only when it began / this, us, causal, batch x sequence, query
// heads on KV heads, head size: 2 x 32 4 on 4 16 12.2 / 5.5; 1 x 448 3 on 3 32 32.5 / 17.2; 16 x 256 8 on 2 32 56.7 / 34.5; 7 x 448
// 4 on 4 64 66.4 / 57.4; 8 x 300 4 on 4 96 66.6 / 56.5; 1 x 800 8 on 8 128 163 / 92; 16 x 200 8 on 8 128 178 / 167 (one wave per
// SIMD, registers full: its items still wait for their rows).
template <int K8, bool FULL>
__global__ __launch_bounds__(64 * kMaxWaves<K8>) void attn_f32_bwd_kernel(AttnArgs a, int kblocks, int wq) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    if ((int)blockIdx.x < kblocks) return bwd_dkv<K8, FULL, false, true>(a, blockIdx.x, wave, nw);
    const int sub = wave / wq;
    bwd_dq<K8, FULL, false, false>(a, ((int)blockIdx.x - kblocks) * (nw / wq) + sub, wave % wq, wq, meet + sub * f32_attn_dq_meet((K8 + 3) / 4, wq));
}
// One after the other: large grids of large heads (F32AttnPlan), and where a result lies over an operand or rows are far apart.
template <int K8, bool FULL, bool FAR>
__global__ __launch_bounds__(64 * kMaxWaves<K8>) void attn_f32_bwd_dq_kernel(AttnArgs a) {
    bwd_dq<K8, FULL, FAR, true>(a, blockIdx.x, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), blockDim.x >> 6, meet);
}
template <int K8, bool FULL, bool FAR>
__global__ __launch_bounds__(64 * kMaxWaves<K8>) void attn_f32_bwd_dkv_kernel(AttnArgs a) {
    bwd_dkv<K8, FULL, FAR, false>(a, blockIdx.x, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), blockDim.x >> 6);
}

template <int K8, bool FULL, bool FAR>
void launch_f32(eisen_ctx* ctx, const AttnArgs& a, bool backward) {
    const F32AttnPlan p = f32_attn_plan(K8, a.B, a.S, a.Hq, a.Hkv);
    if (!backward) {
        attn_f32_fwd_kernel<K8, FULL, FAR><<<dim3((unsigned)p.qblocks), 64 * p.wq, p.fwd_lds, ctx->stream>>>(a);
        return;
    }
    if (FAR || !p.one || eisen_attention_writes_over_operand(a, sizeof(float))) {
        attn_f32_bwd_dq_kernel<K8, FULL, FAR><<<dim3((unsigned)p.qblocks), 64 * p.wq, p.dq_lds, ctx->stream>>>(a);
        attn_f32_bwd_dkv_kernel<K8, FULL, FAR><<<dim3((unsigned)p.kblocks), 64 * p.wk, p.dkv_lds, ctx->stream>>>(a);
        return;
    }
    if constexpr (!FAR) attn_f32_bwd_kernel<K8, FULL><<<dim3((unsigned)(p.kblocks + p.dq_groups)), 64 * p.wk, p.bwd_lds, ctx->stream>>>(a, (int)p.kblocks, p.wq);
}

template <bool FAR>
void launch_f32_by_head_dim(eisen_ctx* ctx, const AttnArgs& a, bool backward) {
    switch (a.hd) {
        case 16: return launch_f32<2, true, FAR>(ctx, a, backward);
        case 32: return launch_f32<4, true, FAR>(ctx, a, backward);
        case 48: return launch_f32<6, true, FAR>(ctx, a, backward);
        case 64: return launch_f32<8, true, FAR>(ctx, a, backward);
        case 80: return launch_f32<10, true, FAR>(ctx, a, backward);
        case 96: return launch_f32<12, true, FAR>(ctx, a, backward);
        case 128: return launch_f32<16, true, FAR>(ctx, a, backward);
    }
    if (a.hd < 16) launch_f32<2, false, FAR>(ctx, a, backward);
    else if (a.hd < 32) launch_f32<4, false, FAR>(ctx, a, backward);
    else if (a.hd < 64) launch_f32<8, false, FAR>(ctx, a, backward);
    else launch_f32<16, false, FAR>(ctx, a, backward);
}

}  // namespace

bool eisen_attention_f32_mfma_supports(const AttnArgs& a) {
    const long long n_t = (a.S + 31) / 32;
    return a.hd <= 128 && n_t * a.Hq * a.B < (1ll << 31);
}

void eisen_attention_launch_f32(eisen_ctx* ctx, const AttnArgs& a, bool backward) {
    if (std::max(std::abs(a.q_ss), std::abs(a.k_ss)) < 1ll << 24) launch_f32_by_head_dim<false>(ctx, a, backward);
    else launch_f32_by_head_dim<true>(ctx, a, backward);
}

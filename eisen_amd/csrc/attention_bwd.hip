// Flash-attention backward, the key-stationary pass: dK and dV (head_dim a multiple of 16 up to 128, bf16 MFMA).
//
//   dV = P^T dO,  dK = scale dS^T Q,  dS = P o (dO V^T - D),  P = exp2(log2e (scale Q K^T - LSE))
// summed over the query heads of a KV group (the repeat_kv backward, src/graph/ops/gqa.rs:168-184) and over every
// query that sees the key (the bmm backward of the reference's chain, src/graph/ops/linear.rs:1482-1498, and the
// softmax backward, src/graph/ops/reduction.rs:504-512).  The reference has no such kernel; what it must equal is
// that chain.
//
// Shape of the kernel
//   * A workgroup owns the keys of two 32-key blocks of one KV head, a heavy one and its light mirror image under the
//     causal mask (equal work everywhere).  Its four waves each take every fourth (query head of the group, 32-query
//     tile) item; their partial dK / dV meet in LDS once per key block, in wave order (no atomics).
//   * A tile is a chain of latencies per wave (loads issued, operand reads, two dependent MFMA groups with the softmax
//     between them) that the second wave of the SIMD covers in part.  So a wave must fit 256 registers (two per SIMD) and
//     should spend as few cycles as possible on anything but MFMAs and the softmax:
//       - every MFMA takes its accumulator in ordinary VGPRs (the file is compiled that way): with the AGPR form the
//         compiler copies the score accumulators between the register files around the softmax of every tile;
//       - Q / dO tiles and the two per-query statistics go from global memory straight into a private two-stage LDS
//         ring of the wave (global_load_lds with a scalar base: no staging registers, no LDS stores, no address
//         arithmetic in vector registers, no barrier in the loop);
//       - the score accumulator starts at -LSE / scale and the dP accumulator at D (read from the ring straight into
//         the accumulator registers), and the sign of V is flipped once per key block, so the MFMA chains deliver
//         S - LSE / scale and D - dP: a probability is one multiply and one exp2, -dS one more multiply; -scale is
//         applied when dK is stored.
//   * head_dim above 64: the accumulators and operands of 32 keys need more than 256 registers and the rings 133 KB of LDS, so
//     there is one wave per SIMD and one workgroup per CU.  dK and dV, which only MFMAs touch inside the loop, then stand in
//     the other half of the register file (AGPRs; left to itself the compiler moves operands and scores back and forth
//     between the halves, 250 moves in the loop), and a workgroup takes one key block where there is more than one pair for
//     every CU, the longest first: two pairs on one CU and one on the next cost a third of the time.
//     1 x 6001 x 16 heads of 128 on 4 KV heads, causal: 445 us; the register-staged kernel this replaced took 708.
#include "attention_dq.cuh"

namespace {

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void mfma(f32x16& acc, const bf16x8& a, const bf16x8& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}

// The same with the accumulator in AGPRs.  The compiler does not see an MFMA here, so what it would keep apart is kept apart by
// hand: two wait states between the vector instruction that wrote an operand and the MFMA, and agpr_settle() between the
// last MFMA and the first other reader of the accumulators.  No copy and no spill of an accumulator may stand in the loop or
// before the settling: the build reads the assembly and fails if one does (check_agpr_loops.py).
__device__ __forceinline__ void mfma_agpr(f32x16& acc, const bf16x8& a, const bf16x8& b) {
    asm("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void agpr_settle(f32x16& acc) { asm volatile("s_nop 15\n\ts_nop 7" : "+a"(acc)); }

// ABL: a part of the tile loop left out for a measurement (AttnAblation; kAblNone is the kernel)
// GW > 0: short sequences, both passes side by side in one launch, the first dq_blocks workgroups on dQ (with GW query heads to a workgroup).  One after the other they are
// two latencies and a launch, with much of the chip idle: 4 x 256 tokens, 16 heads of 64, dQ 12.3 us and dK / dV 8.3.  The workgroups of this pass compute the
// statistics that the dQ pass would have left them (the results are the same to the bit), which takes them 1 to 2 us where they see 8 to 16
// query tiles.  Where it is used, and what it takes: eisen_attention_bwd_short_supports.
constexpr int kOwnTiles = 64;  // places for the statistics of a tile, behind the rings
template <int HD>
struct DqLds {
    __attribute__((aligned(1024))) bf16_t k[kDqTiles<HD>];
    __attribute__((aligned(1024))) bf16_t v[kDqTiles<HD>];
    __attribute__((aligned(1024))) bf16_t rows[kDqRows<HD, kAblNone>];
};
// ONE: a workgroup takes one key block, not a pair (key_blocks_paired; head sizes above 64 have a.kb_paired in launches of their own).
template <int HD, int ABL, int GW = 0, bool ONE = false>
__global__ __launch_bounds__(256, HD <= 64 ? 2 : 1) void fa_bwd_dkv32_kernel(AttnArgs a) {
    constexpr bool OWN = GW > 0;
    constexpr int KSTEPS = HD / 16, DT = (HD + 31) / 32, NST = 2;
    constexpr int TILE = 32 * kTileRow<HD>;                          // elements of a Q or dO tile
    constexpr int STAGE_BYTES = 2 * TILE * 2 + (OWN ? 0 : 256);      // Q tile, dO tile, 32 x (-LSE / scale | D)
    // dK and dV in AGPRs (not beside the dQ role, where the compiler reads the accumulators before the wait states; in short loops its moves matter less)
    constexpr bool AGPR = HD > 64 && !OWN;
    using Loader = DirectTile<HD, 32, 1>;
    constexpr int LOADS = 2 * Loader::PER_WAVE + 1;      // load instructions per tile
    static_assert(LOADS <= 63, "the tile in flight must fit the vmcnt counter");
    static_assert(2 * 4 * 32 * HD * sizeof(float) <= 4 * NST * STAGE_BYTES, "the reduction of dK and dV reuses the rings");
    constexpr int RINGS = 4 * NST * STAGE_BYTES, BYTES = !OWN ? RINGS : RINGS + kOwnTiles * 256 > (int)sizeof(DqLds<HD>) ? RINGS + kOwnTiles * 256 : (int)sizeof(DqLds<HD>);
    static_assert(!OWN || BYTES <= (HD <= 64 ? 80 : 160) * 1024, "two workgroups per CU, one for the head sizes above 64");
    __shared__ __attribute__((aligned(1024))) char lds[BYTES];
    int block = blockIdx.x, blocks = gridDim.x;
    if constexpr (OWN) {
        if (block < a.dq_blocks) {
            DqLds<HD>& dq = *reinterpret_cast<DqLds<HD>*>(lds);
            bwd_dq<HD, GW, kAblNone, false>(a, dq.k, dq.v, dq.rows, block, a.dq_blocks);
            return;
        }
        block -= a.dq_blocks;
        blocks -= a.dq_blocks;
    }

    const int lane = threadIdx.x & 63, g = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_qt = (a.S + 31) / 32, n_pairs = (n_qt + 1) / 2;
    // grid: x = key-block pair, fastest; then KV head, then batch.  Blocks of one (batch, KV head) read the same
    // Q / dO tiles, so they are kept on one XCD.
    // Without pairs: the key block slowest, longest (causal) first.
    const bool paired = !ONE && (HD <= 64 || OWN || a.kb_paired);
    const int bid = paired ? xcd_contiguous_id(block, blocks) : block;
    const int pair = paired ? bid % n_pairs : bid / (a.Hkv * a.B), of = paired ? bid / n_pairs : bid % (a.Hkv * a.B);
    const int kvh = of % a.Hkv, b = of / a.Hkv;
    char* ring = lds + wave * (NST * STAGE_BYTES);
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    // lanes 0-31 fetch the tile's -LSE / scale, lanes 32-63 its D: byte offset of the lane's value from D's entry for the
    // tile's first query (the launcher has checked that the statistics are less than 2 GiB apart)
    const unsigned stat_off = (unsigned)(g == 0 ? (a.L2 - a.D) * 4 : 0) + 4 * (unsigned)c;
    float* const own = reinterpret_cast<float*>(lds + (OWN ? RINGS : 0));  // OWN: [query head of the group][query tile from own_first]
    const int own_first = a.causal ? pair : 0, own_per_head = n_qt - own_first;
    Loader loader;
    loader.init(a.q_ss, 0, lane);
    constexpr bool TL = ABL == kAblTimeline;
    attn_stamp<TL>(a, 2, kStampStart, lane, wave);

    // K and V rows of this lane's key of key block kb_, as they are stored
    bf16x8 kraw[KSTEPS], vraw[KSTEPS];
    auto load_kv = [&](int kb_) {
        const int key_ = kb_ * 32 + c;
        const long long koff = b * a.k_sb + kvh * a.k_sh + (long long)key_ * a.k_ss;
#pragma unroll
        for (int st = 0; st < KSTEPS; st++) {
            const int d = st * 16 + 8 * g;
            kraw[st] = key_ < a.S ? *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.K) + koff + d) : zero8;
            vraw[st] = key_ < a.S ? *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.V) + koff + d) : zero8;
        }
    };

    if constexpr (OWN) {
        // The statistics of every tile that these keys see (of the second pass's as well: a part of them), as the dQ pass computes them, the loads
        // of U tiles at a time in flight.
        constexpr int U = HD <= 32 ? 8 : HD <= 64 ? 4 : 2;
        const int tiles = a.G * own_per_head;
        for (int t0 = wave; t0 < tiles; t0 += 4 * U) {
            bf16x8 x[U][KSTEPS], y[U][KSTEPS];
            float lse[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = t0 + 4 * u;
                if (t >= tiles) break;
                const int head = t / own_per_head, row = min((own_first + t - head * own_per_head) * 32 + c, a.S - 1);
                const long long at = b * a.q_sb + (kvh * a.G + head) * a.q_sh + (long long)row * a.q_ss + 8 * g;
#pragma unroll
                for (int st = 0; st < KSTEPS; st++) {
                    x[u][st] = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.dO) + at + st * 16);
                    y[u][st] = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.O) + at + st * 16);
                }
                lse[u] = a.LSE[((long long)b * a.Hq + kvh * a.G + head) * a.S + row];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = t0 + 4 * u;
                if (t >= tiles) break;
                float part = 0.f;
#pragma unroll
                for (int st = 0; st < KSTEPS; st++)
#pragma unroll
                    for (int e = 0; e < 8; e++) part += (float)x[u][st][e] * (float)y[u][st][e];
                const float sum = part + __shfl_xor(part, 32, 64);
                const bool past = (own_first + t % own_per_head) * 32 + c >= a.S;  // a query past the end: probabilities exactly zero
                own[t * 64 + lane] = g ? sum : past ? -INFINITY : -lse[u] / a.scale;
            }
        }
        __syncthreads();
    }

    for (int pass = 0; pass < 2; pass++) {
        const int kb = pass == 0 ? pair : n_qt - 1 - pair;
        if (pass == 1 && (!paired || kb <= pair)) break;  // odd block count: the middle block has no mirror
        const int k0 = kb * 32;
        if (pass == 0) load_kv(kb);  // the second pass's rows were requested before the first pass's reduction
        f32x16 dk[DT], dv[DT];
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) { dk[dt][v] = 0.f; dv[dt][v] = 0.f; }

        const int qt_start = a.causal ? kb : 0;  // the diagonal tile is the first one that sees these keys
        const int per_head = n_qt - qt_start;
        const int n_items = a.G * per_head;       // (query head of the group, query tile), head-major
        const int n_mine = n_items > wave ? (n_items - wave + 3) / 4 : 0;

        auto stage_of = [&](int i) { return ring + (ABL == kAblTileLoads ? 0 : (i % NST)) * STAGE_BYTES; };
        // The tile that the next issue() requests, kept as running sums (all wave-uniform, so scalar registers): this wave's
        // items are wave, wave + 4, ... in head-major order; a step of four tiles that runs past the head's last tile
        // wraps into the next head.
        int nrel = wave % per_head;                    // tile index within the head, from the diagonal tile
        int nq0 = (qt_start + nrel) * 32;              // its first query
        long long ntile, nstat;                        // element offsets of its Q / dO rows and of its statistics
        {
            const int hq = kvh * a.G + wave / per_head;
            ntile = b * a.q_sb + hq * a.q_sh + (long long)nq0 * a.q_ss;
            nstat = ((long long)b * a.Hq + hq) * a.S + nq0;
        }
        int nown = wave / per_head * own_per_head + qt_start - own_first + nrel;  // OWN: its place
        const long long tile_wrap = a.q_sh - (long long)per_head * 32 * a.q_ss, stat_wrap = (long long)a.S - per_head * 32;
        auto issue = [&](int i) -> int {  // the loads of this wave's i-th tile into ring stage i % NST; returns the tile's first query
            const int q0 = nq0;
            char* stage = stage_of(i);
            const char* qbase = reinterpret_cast<const char*>(static_cast<const bf16_t*>(a.Q) + ntile);
            const char* dobase = reinterpret_cast<const char*>(static_cast<const bf16_t*>(a.dO) + ntile);
            const char* sbase = reinterpret_cast<const char*>(a.D + nstat);
            nrel += 4; nq0 += 128; ntile += 128 * a.q_ss; nstat += 128; nown += 4;
            while (nrel >= per_head) { nrel -= per_head; nq0 -= per_head * 32; ntile += tile_wrap; nstat += stat_wrap; nown += own_per_head - per_head; }
            if (q0 + 32 <= a.S) {
#pragma unroll
                for (int r = 0; r < Loader::PER_WAVE; r++) {
                    load_lds_16(qbase, loader.off[r], stage + r * 1024);
                    load_lds_16(dobase, loader.off[r], stage + TILE * 2 + r * 1024);
                }
                if (!OWN) load_lds_4(sbase, stat_off, stage + 2 * TILE * 2);
            } else {  // ragged last tile: rows past the end re-read the last row (they are given zero weight)
#pragma unroll
                for (int r = 0; r < Loader::PER_WAVE; r++) {
                    const int row = Loader::lane_row(0, r, lane), gr = min(row, a.S - 1 - q0);
                    const unsigned off = (unsigned)((gr * a.q_ss + Loader::lane_chunk(row, lane) * 8) * 2);
                    load_lds_16(qbase, off, stage + r * 1024);
                    load_lds_16(dobase, off, stage + TILE * 2 + r * 1024);
                }
                if (!OWN) load_lds_4(sbase, stat_off - 4 * (unsigned)(c - min(c, a.S - 1 - q0)), stage + 2 * TILE * 2);
            }
            return q0;
        };

        int own_next = nown;
        int q0_next = n_mine > 0 ? issue(0) : 0;
        bf16x8 kf[KSTEPS], vn[KSTEPS];  // K and -V of the 32 keys, MFMA B operands (requested before the first tile, used after it is)
#pragma unroll
        for (int st = 0; st < KSTEPS; st++) {
            typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
            kf[st] = kraw[st];
            u32x4 bits = __builtin_bit_cast(u32x4, vraw[st]) ^ 0x80008000u;  // sign flip of the eight bf16 values
            vn[st] = __builtin_bit_cast(bf16x8, bits);
            // the flip is done here, once, not again at every use; and both operands have arrived before the loop (a
            // pending load of theirs would make the compiler wait for every outstanding load at their first use in it,
            // the prefetched tile's included)
            asm volatile("" : "+v"(vn[st]), "+v"(kf[st]));
        }
        attn_stamp<TL>(a, 2, kStampLoop + kStampsPerPass * pass, lane, wave);
        for (int i = 0; i < n_mine; i++) {
            wait_vmcnt<0>();  // tile i was requested in the middle of tile i - 1
            const int q0 = q0_next;
            const bf16_t* Qs = reinterpret_cast<const bf16_t*>(stage_of(i));
            const bf16_t* dOs = Qs + TILE;
            float* st = OWN ? own + own_next * 64 : reinterpret_cast<float*>(stage_of(i) + 2 * TILE * 2);
            if (!OWN && q0 + 32 > a.S) {  // a query past the end gets LSE = +inf (stored negated): its probabilities are exactly zero
                if (g == 0 && q0 + c >= a.S) st[c] = -INFINITY;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            // scores: S - LSE / scale and D - dP, the start values read straight into the accumulator registers
            f32x16 s, dp;
#pragma unroll
            for (int vg = 0; vg < 4; vg++) {
                const float4 l4 = *reinterpret_cast<const float4*>(st + 8 * vg + 4 * g);
                const float4 d4 = *reinterpret_cast<const float4*>(st + 32 + 8 * vg + 4 * g);
                s[4 * vg] = l4.x; s[4 * vg + 1] = l4.y; s[4 * vg + 2] = l4.z; s[4 * vg + 3] = l4.w;
                dp[4 * vg] = d4.x; dp[4 * vg + 1] = d4.y; dp[4 * vg + 2] = d4.z; dp[4 * vg + 3] = d4.w;
            }
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ks++) {
                const bf16x8 qa = ABL == kAblOperandReads ? vn[ks] : *reinterpret_cast<const bf16x8*>(Qs + tile_at<HD>(c, ks * 16 + 8 * g));
                const bf16x8 da = ABL == kAblOperandReads ? kf[ks] : *reinterpret_cast<const bf16x8*>(dOs + tile_at<HD>(c, ks * 16 + 8 * g));
                if (ABL == kAblScoreMfmas) { s[ks] += (float)qa[0]; dp[ks] += (float)da[0]; }
                else {
                mfma(s, qa, kf[ks]);
                mfma(dp, da, vn[ks]);
                }
            }
            // the transposed operands of the accumulation, requested before the softmax so that they arrive under it
            bf16x8 dotr[DT][2], qtr[DT][2];
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    if (ABL == kAblTransposedReads) { dotr[dt][t] = kf[dt * 2 + t]; qtr[dt][t] = vn[dt * 2 + t]; }
                    else {
                    dotr[dt][t] = lds_tr_operand_swz<HD>(dOs, 0, dt * 32, t, lane);
                    qtr[dt][t] = lds_tr_operand_swz<HD>(Qs, 0, dt * 32, t, lane);
                    }
                }
            // the next tile's loads go out while the score MFMAs run (the other stage was read by tile i - 1, whose operand reads
            // have all returned)
            own_next = nown;
            if (ABL != kAblTileLoads && i + 1 < n_mine) q0_next = issue(i + 1);
            float p[16];
#pragma unroll
            for (int v = 0; v < 16; v++) p[v] = ABL == kAblSoftmax ? s[v] : fast_exp2(s[v] * a.scale_log2e);
            // only the diagonal tile is cut by the causal mask
            if (a.causal && q0 == k0) {
                asm volatile("" ::: "memory");  // keeps this a branch taken once per head, not 16 selects per tile
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (c > acc_row(v, g)) p[v] = 0.f;  // key k0 + c is after query q0 + row
            }
            bf16x8 pf[2], dsf[2];
#pragma unroll
            for (int v = 0; v < 16; v++) {
                pf[v >> 3][v & 7] = (bf16_t)p[v];
                dsf[v >> 3][v & 7] = (bf16_t)(ABL == kAblSoftmax ? dp[v] : p[v] * dp[v]);  // = -dS: dp holds D - dP
            }
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    if (ABL == kAblSecondMfmas) { dv[dt][0] += (float)pf[t][0] * (float)dotr[dt][t][0]; dk[dt][0] += (float)dsf[t][0] * (float)qtr[dt][t][0]; }
                    else {
                    if (AGPR) {
                        mfma_agpr(dv[dt], pf[t], dotr[dt][t]);
                        mfma_agpr(dk[dt], dsf[t], qtr[dt][t]);
                    } else {
                        mfma(dv[dt], pf[t], dotr[dt][t]);
                        mfma(dk[dt], dsf[t], qtr[dt][t]);
                    }
                    }
                }
        }
        if (AGPR) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++) { agpr_settle(dv[dt]); agpr_settle(dk[dt]); }
        }
        attn_stamp<TL>(a, 2, kStampLoopEnd + kStampsPerPass * pass, lane, wave);
        // the mirror block's K and V rows travel while this block's partial results are summed
        if (pass == 0 && paired && n_qt - 1 - pair > pair) load_kv(n_qt - 1 - pair);
        // Sum the four waves' partial results through the (now idle) rings and store: dK and dV in one round.
        float* red = reinterpret_cast<float*>(lds);  // [dK | dV][wave][32 keys][HD]
        bf16_t* outs[2] = {static_cast<bf16_t*>(a.dK) + b * a.k_sb + kvh * a.k_sh, static_cast<bf16_t*>(a.dV) + b * a.k_sb + kvh * a.k_sh};
        __syncthreads();  // every wave is done with its ring
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int at = (wave * 32 + acc_row(v, g)) * HD + dt * 32 + c;
                if (dt * 32 + 32 > HD && dt * 32 + c >= HD) continue;
                red[at] = dk[dt][v] * -a.scale;
                red[4 * 32 * HD + at] = dv[dt][v];
            }
        __syncthreads();
#pragma unroll
        for (int which = 0; which < 2; which++) {
            for (int e0 = threadIdx.x * 8; e0 < 32 * HD; e0 += 256 * 8) {
                float acc8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < 4; w++) {
                    const float* src = red + (which * 4 + w) * 32 * HD + e0;
                    const float4 x0 = *reinterpret_cast<const float4*>(src);
                    const float4 x1 = *reinterpret_cast<const float4*>(src + 4);
                    acc8[0] += x0.x; acc8[1] += x0.y; acc8[2] += x0.z; acc8[3] += x0.w;
                    acc8[4] += x1.x; acc8[5] += x1.y; acc8[6] += x1.z; acc8[7] += x1.w;
                }
                const int kr = k0 + e0 / HD;
                if (kr < a.S) {
                    if (which == 0 && a.rope) unrotate_pairs<4>(acc8, a.rope + (size_t)kr * (HD / 2) + (e0 % HD) / 2);
                    bf16x8 o8;
#pragma unroll
                    for (int e = 0; e < 8; e++) o8[e] = (bf16_t)acc8[e];
                    *reinterpret_cast<bf16x8*>(outs[which] + (long long)kr * a.k_ss + e0 % HD) = o8;
                }
            }
        }
        __syncthreads();  // the reduction's reads are over before the next pass refills the rings
        attn_stamp<TL>(a, 2, kStampStored + kStampsPerPass * pass, lane, wave);
    }
}

}  // namespace

// What the kernel above covers: shapes whose byte offsets inside a tile (31 rows of the query
// stride) and between the two statistics arrays fit 32 bits.
bool eisen_attention_dkv32_supports(const AttnArgs& a) {
    return a.hd <= 128 && a.hd % 16 == 0 && a.q_ss > 0 && a.q_ss * 32 * 2 < (1ll << 31) && a.L2 > a.D && (a.L2 - a.D) * 4 < (1ll << 31);
}

// Whether a result lies over an operand, or dQ is where dK or dV is.  In two launches dQ may take the place of O, and dK and dV that of K, V or O, which nobody reads any more by
// then; in one they are still being read.
bool eisen_attention_writes_over_operand(const AttnArgs& a, size_t element) {
    struct Range {
        const void* from;
        size_t bytes;
    };
    auto range = [&](const void* p, int heads, long long sb, long long ss, long long sh) {
        long long lowest = 0, end = a.hd;
        for (const long long reach : {(a.B - 1) * sb, (a.S - 1) * ss, (heads - 1) * sh}) (reach < 0 ? lowest : end) += reach;
        return Range{static_cast<const char*>(p) + lowest * (long long)element, (size_t)(end - lowest) * element};
    };
    auto q = [&](const void* p) { return range(p, a.Hq, a.q_sb, a.q_ss, a.q_sh); };
    auto k = [&](const void* p) { return range(p, a.Hkv, a.k_sb, a.k_ss, a.k_sh); };
    for (const Range& out : {q(a.dQ), k(a.dK), k(a.dV)})
        for (const Range& in : {q(a.Q), k(a.K), k(a.V), q(a.O), q(a.dO), Range{a.LSE, sizeof(float) * a.B * a.Hq * a.S}})
            if (eisen_ranges_meet(out.from, out.bytes, in.from, in.bytes)) return true;
    return a.dQ == a.dK || a.dQ == a.dV;
}

// Whether a dK / dV workgroup takes two key blocks, a long one and its short mirror image (for equal work), or one: where there are places for all of
// them at once (two workgroups to a CU; one for head sizes above 64), beside those of the dQ pass that share the launch, the pair would only be done one after the
// other.  The results are the same to the bit.  Backward with pairs / without, us, batch x sequence, query heads on KV heads, head size: 10 x 44 8 on 8 64 7.9 / 6.2; 1 x
// 130 3 on 3 64 9.2 / 7.2; 7 x 193 6 on 6 48 8.9 / 8.1; 1 x 506 4 on 2 64 20.6 / 18.2; 3 x 512 8 on 8 64 16.2 / 14.2; 2 x 1000 6 on 6 64 24.7 / 21.3; 1 x 512 8 on 4
// 96 30.1 / 26.3; 1 x 2048 2 on 2 128 61.8 / 57.2; in two launches 2 x 448 9 on 3 80 34.2 / 29.2; 7 x 668 6 on 3 64 30.0 / 30.0.  (Of 89 shapes at random that go one by one 7 lose by it, 2 % at most,
// 1 x 3590 16 on 4 64 140.8 / 143.2; the median gains 13 %.)
static bool key_blocks_paired(const AttnArgs& a, int dq_blocks) { return dq_blocks + (long long)((a.S + 31) / 32) * a.Hkv * a.B > (a.hd <= 64 ? 512 : 256); }

// Where one launch (fa_bwd_dkv32_kernel with GW > 0) takes less time than two: where every workgroup is on the chip at once, two to a CU (head sizes above 64: one), and a
// workgroup of the dK / dV role has few enough statistics to compute before it starts.  With larger query groups there are fewer of these
// workgroups, each with more tiles, and the statistics come on top of what was the longer pass already.  Two launches / one, us, causal, batch x sequence,
// query heads on KV heads, head size: 4 x 256 16 on 16 64 16.1 / 12.9; 7 x 193 6 on 6 48 14.7 / 8.7; 1 x 2048 8 on 8 64 49.6 / 39.7; 4 x 512 8 on 4 128 45.1 /
// 38.3; 4 x 256 8 on 8 128 30.6 / 19.4.  Beyond the lines: 8 x 256 16 on 16 64 (768 workgroups) 20.2 / 20.6, 16 x 256 33.0 / 37.9; 4 x 256 24 on 8 64 19.3 / 19.8;
// 1 x 512 32 on 8 64 28.6 / 33.4; 1 x 512 16 on 4 128 53.5 / 61.2; 2 x 256 32 on 4 64 26.2 / 34.2.  At them: 8 x 128 8 on 2 64 15.3 / 13.9; 21 x 256 8 on 2 32 17.6 / 16.2;
// 8 x 256 8 on 2 48 19.0 / 18.1; 4 x 64 16 on 2 64 15.2 / 14.6; 1 x 1024 16 on 8 64 35.3 / 34.1.
// Three query heads on a KV head, no pairs of key blocks: up to 64 tiles where the head size is no multiple of 64 (1 x 672 3 on 1 16 20.1 / 14.0; 1 x 512 24 on 8 32 18.4 / 16.8; 3 x
// 500 6 on 2 48 22.2 / 17.7; 2 x 448 9 on 3 80 29.1 / 23.7, 96 30.6 / 27.0, 112 36.4 / 31.4; 2 x 672 9 on 3 96 41.1 / 36.9, 112 48.2 / 43.2; 1 x 448 24 on 8 96 31.2 / 31.6; 1 x 672 24 on 8
// 48 26.0 / 26.8), half as many where it is (2 x 250 9 on 3 64 16.4 / 14.8, 128 30.4 / 25.3; but 2 x 448 64 21.4 / 22.5, 128 38.4 / 40.5; 2 x 672 64 27.8 / 30.9, 128 50.7 / 56.6; why those
// two sizes gain less is not known: their one launch takes about as long as that of the next larger size, 2 x 512 9 on 3 64 24.8 beside 26.4 for 80).
bool eisen_attention_bwd_short_supports(const AttnArgs& a, int dq_blocks) {
    const int n_qt = (a.S + 31) / 32;
    const bool three = a.G == 3 && !key_blocks_paired(a, dq_blocks);
    const int most = a.G <= 2 || (three && a.hd % 64 != 0) ? kOwnTiles : three || (a.G <= 4 && a.hd != 64) ? 32 : 16;
    const long long blocks = dq_blocks + (long long)(n_qt + 1) / 2 * a.Hkv * a.B;
    return a.G * n_qt <= most && blocks <= (a.hd <= 64 ? 512 : 256) && a.ablation == kAblNone && eisen_attention_dkv32_supports(a) && !eisen_attention_writes_over_operand(a, 2);
}

void eisen_attention_launch_bwd_short(eisen_ctx* ctx, AttnArgs a, int gw, int dq_blocks) {
    a.dq_blocks = dq_blocks;
    a.kb_paired = key_blocks_paired(a, dq_blocks);
    const int blocks = dq_blocks + (a.kb_paired ? ((a.S + 31) / 32 + 1) / 2 : (a.S + 31) / 32) * a.Hkv * a.B;
    auto launch = [&](auto hd) {
        constexpr int HD = decltype(hd)::value;
        auto as = [&](auto one_c) {
            constexpr bool ONE = decltype(one_c)::value;
            if (gw == 4) fa_bwd_dkv32_kernel<HD, kAblNone, 4, ONE><<<blocks, 256, 0, ctx->stream>>>(a);
            else if (gw == 2) fa_bwd_dkv32_kernel<HD, kAblNone, 2, ONE><<<blocks, 256, 0, ctx->stream>>>(a);
            else fa_bwd_dkv32_kernel<HD, kAblNone, 1, ONE><<<blocks, 256, 0, ctx->stream>>>(a);
        };
        if (a.kb_paired) as(std::false_type{});
        else as(std::true_type{});
    };
    switch (a.hd) {
        case 16: return launch(std::integral_constant<int, 16>{});
        case 32: return launch(std::integral_constant<int, 32>{});
        case 48: return launch(std::integral_constant<int, 48>{});
        case 64: return launch(std::integral_constant<int, 64>{});
        case 80: return launch(std::integral_constant<int, 80>{});
        case 96: return launch(std::integral_constant<int, 96>{});
        case 112: return launch(std::integral_constant<int, 112>{});
        default: return launch(std::integral_constant<int, 128>{});
    }
}

// a.L2 (-LSE / scale) and a.D must have been written (by the dQ kernel).
void eisen_attention_launch_dkv32(eisen_ctx* ctx, AttnArgs a) {
    const int n_kb = (a.S + 31) / 32;  // 32-key blocks, handled in heavy / light pairs or one by one
    const long long pairs = (long long)(n_kb + 1) / 2 * a.Hkv * a.B;
    a.kb_paired = (a.hd <= 64 || pairs <= 256) && (a.ablation != kAblNone || key_blocks_paired(a, 0));
    dim3 grid((unsigned)(a.kb_paired ? pairs : (long long)n_kb * a.Hkv * a.B));
    if (a.hd == 64 && (a.kb_paired || a.ablation != kAblNone)) {
        switch (a.ablation) {  // hd 64 only: the head size the measurements are quoted for
            case kAblTransposedReads: fa_bwd_dkv32_kernel<64, kAblTransposedReads><<<grid, 256, 0, ctx->stream>>>(a); break;
            case kAblOperandReads: fa_bwd_dkv32_kernel<64, kAblOperandReads><<<grid, 256, 0, ctx->stream>>>(a); break;
            case kAblSecondMfmas: fa_bwd_dkv32_kernel<64, kAblSecondMfmas><<<grid, 256, 0, ctx->stream>>>(a); break;
            case kAblTileLoads: fa_bwd_dkv32_kernel<64, kAblTileLoads><<<grid, 256, 0, ctx->stream>>>(a); break;
            case kAblSoftmax: fa_bwd_dkv32_kernel<64, kAblSoftmax><<<grid, 256, 0, ctx->stream>>>(a); break;
            case kAblScoreMfmas: fa_bwd_dkv32_kernel<64, kAblScoreMfmas><<<grid, 256, 0, ctx->stream>>>(a); break;
            case kAblTimeline: fa_bwd_dkv32_kernel<64, kAblTimeline><<<grid, 256, 0, ctx->stream>>>(a); break;
            default: fa_bwd_dkv32_kernel<64, kAblNone><<<grid, 256, 0, ctx->stream>>>(a); break;
        }
    }
    else if (a.hd == 128) fa_bwd_dkv32_kernel<128, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 112) fa_bwd_dkv32_kernel<112, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 96) fa_bwd_dkv32_kernel<96, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 80) fa_bwd_dkv32_kernel<80, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 64) fa_bwd_dkv32_kernel<64, kAblNone, 0, true><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 48 && a.kb_paired) fa_bwd_dkv32_kernel<48, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 48) fa_bwd_dkv32_kernel<48, kAblNone, 0, true><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 32 && a.kb_paired) fa_bwd_dkv32_kernel<32, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.hd == 32) fa_bwd_dkv32_kernel<32, kAblNone, 0, true><<<grid, 256, 0, ctx->stream>>>(a);
    else if (a.kb_paired) fa_bwd_dkv32_kernel<16, kAblNone><<<grid, 256, 0, ctx->stream>>>(a);
    else fa_bwd_dkv32_kernel<16, kAblNone, 0, true><<<grid, 256, 0, ctx->stream>>>(a);
}

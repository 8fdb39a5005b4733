// The query-stationary half of the attention backward, dQ, and the order of the blocks of the two query-stationary passes: a kernel of its own in attention.hip, one
// role of the one that takes both passes in attention_bwd.hip.
#pragma once
#include "attention_common.cuh"

namespace {

// Grid of the two query-stationary kernels: one block per (pair of query blocks, GW query heads of a
// KV head, batch), pair index fastest.  A block runs query block `pair` and then its mirror image
// n-1-pair, so that under the causal mask every block sees the same number of key tiles; blocks that
// read the same K/V (one batch and KV head) are kept on one XCD.
struct QBlock {
    int pair, n_qblk, kvh, hgrp, b;
};
template <int GW>
__device__ __forceinline__ QBlock decode_qblock(const AttnArgs& a, int block, int blocks) {
    constexpr int QS = 4 / GW;
    QBlock r;
    r.n_qblk = (a.S + 32 * QS - 1) / (32 * QS);
    const int n_pairs = a.paired ? (r.n_qblk + 1) / 2 : r.n_qblk, groups = a.G / GW;
    // Blocks of one (batch, KV head) on one XCD.  Unpaired blocks differ in length under the causal mask: the longest ones are
    // started first (pair index slowest in launch order), so that the short ones fill the end.  Workgroups go to the XCDs in
    // turn, so with the groups fastest a group keeps to its XCDs where their number divides 8 (and with 8 n groups every XCD
    // has n); other numbers spread a group over the XCDs, which costs less than XCDs of long and of short blocks only.  Without the
    // mask all blocks are equal and a group keeps to its XCD whatever the number of groups (spread / kept, forward + backward, us:
    // 11 x 1024, 12 heads on 3, 55.5 + 187.1 / 52.2 + 180.5; 3 x 4096, 5 of 128, 149.0 + 539.9 / 142.5 + 532.8; level at few blocks).
    int bid;
    const int per = blocks / 8;
    if (!a.paired && blocks % 8 == 0 && per % n_pairs == 0) {
        const int gx = per / n_pairs, xcd = block % 8, local = block / 8;  // gx groups of n_pairs blocks per XCD
        bid = (xcd * gx + local % gx) * n_pairs + local / gx;
    } else if (!a.paired && a.causal) {
        const int all = blocks / n_pairs;
        bid = (block % all) * n_pairs + block / all;
    } else {
        bid = xcd_contiguous_id(block, blocks);
    }
    r.pair = bid % n_pairs;
    const int y = (bid / n_pairs) % (a.Hkv * groups);
    r.kvh = y / groups;
    r.hgrp = y % groups;
    r.b = bid / (n_pairs * a.Hkv * groups);
    return r;
}

// ---- backward: dQ (query-stationary); also writes D = rowsum(dO o O) for the dK/dV pass ------
// ABL: a part of the tile loop left out for a measurement (AttnAblation; kAblNone is the kernel)
//
// A block runs a long query block and then its short mirror image.  For head sizes up to 64 the two are one stream of
// K / V tiles through the two LDS buffers (the short block's first tile is requested under the long block's last one), and
// the rows of Q, dO and O of a wave's 32 queries arrive through three private LDS tiles of the wave, in whole rows; those of
// the short block are requested while the long block's tile loop runs, so that its start-up costs no trip to memory.
// STATS: D and -LSE / scale are stored for a dK / dV kernel that follows.
template <int HD, int ABL>
constexpr bool kDqStream = HD <= 64 && ABL != kAblTileLoads;
// LDS, in elements: the K (V) tiles, and the rows
template <int HD>
constexpr int kDqTiles = 2 * 64 * kTileRow<HD>;
template <int HD, int ABL>
constexpr int kDqRows = kDqStream<HD, ABL> ? 4 * 3 * 32 * kTileRow<HD> : 8;
template <int HD, int GW, int ABL, bool STATS>
__device__ __forceinline__ void bwd_dq(const AttnArgs& a, bf16_t (&Ksb)[kDqTiles<HD>], bf16_t (&Vsb)[kDqTiles<HD>], bf16_t (&Rows)[kDqRows<HD, ABL>], int block, int blocks) {
    constexpr int QS = 4 / GW, BKV = 64, KSTEPS = HD / 16, DT = (HD + 31) / 32;
    constexpr bool STREAM = kDqStream<HD, ABL>;
    constexpr int ROWS = 32 * kTileRow<HD>;  // elements of a wave's Q, dO or O rows
    constexpr int KV = BKV * kTileRow<HD>;   // of a K or V tile: two swizzled tiles of each (see DirectTile); Rows: [wave][Q | dO | O], swizzled like them
    const int lane = threadIdx.x & 63, g = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hsub = wave % GW, qsub = wave / GW;
    const QBlock blk = decode_qblock<GW>(a, block, blocks);
    const int kvh = blk.kvh, hq = kvh * a.G + blk.hgrp * GW + hsub, b = blk.b;
    const bf16_t* Kp = static_cast<const bf16_t*>(a.K) + b * a.k_sb + kvh * a.k_sh;
    const bf16_t* Vp = static_cast<const bf16_t*>(a.V) + b * a.k_sb + kvh * a.k_sh;
    const long long head_off = b * a.q_sb + hq * a.q_sh;
    const long long head_stat = ((long long)b * a.Hq + hq) * a.S;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    DirectTile<HD, BKV, 4> kv_tile;
    kv_tile.init(a.k_ss, wave, lane);
    DirectTile<HD, 32, 1> row_tile;
    if (STREAM) row_tile.init(a.q_ss, 0, lane);
    constexpr bool TL = ABL == kAblTimeline;
    attn_stamp<TL>(a, 1, kStampStart, lane, wave);
    bf16_t* my_rows = Rows + (STREAM ? wave * 3 * ROWS : 0);
    // the rows of Q, dO and O of this wave's queries of query block qb, straight into the wave's LDS tiles (rows past the
    // end repeat the last row; their queries get LSE = +inf below)
    auto request_rows = [&](int qb) {
        const int first = (qb * QS + qsub) * 32;
        row_tile.load_untracked(static_cast<const bf16_t*>(a.Q) + head_off, a.q_ss, first, a.S, my_rows, 0, lane);
        row_tile.load_untracked(static_cast<const bf16_t*>(a.dO) + head_off, a.q_ss, first, a.S, my_rows + ROWS, 0, lane);
        row_tile.load_untracked(static_cast<const bf16_t*>(a.O) + head_off, a.q_ss, first, a.S, my_rows + 2 * ROWS, 0, lane);
    };
    const int qblk_long = blk.n_qblk - 1 - blk.pair, qblk_short = blk.pair;
    const bool two = a.paired && qblk_short < qblk_long;  // the middle block has no mirror
    float lse_short = 0.f;  // STREAM: the short block's LSE, requested with the long block's
    if (STREAM) {
        kv_tile.load_untracked(Kp, a.k_ss, 0, a.S, Ksb, wave, lane);
        kv_tile.load_untracked(Vp, a.k_ss, 0, a.S, Vsb, wave, lane);
        request_rows(qblk_long);
        const int qs = (qblk_short * QS + qsub) * 32 + c;
        if (two && qs < a.S) lse_short = a.LSE[head_stat + qs];
    }
    int par = 0;  // STREAM: LDS buffer of the pass's first K / V tile

    for (int pass = 0; pass < 2; pass++) {
        const int qblk = pass == 0 ? qblk_long : qblk_short;
        if (pass == 1 && !two) break;
        const int q0 = (qblk * QS + qsub) * 32, q = q0 + c;
        const bool valid_q = q < a.S;
        const long long qoff = head_off + (long long)q * a.q_ss;
        const long long stat = head_stat + q;
        bf16x8 qf[KSTEPS], dof[KSTEPS];
        float dpart = 0.f, lse = 0.f;
        if (STREAM) {
            if (pass == 0) lse = valid_q ? a.LSE[stat] : 0.f;
            else lse = lse_short;
            wait_direct_loads();  // this wave's rows have landed (they are private to the wave: no barrier)
#pragma unroll
            for (int st = 0; st < KSTEPS; st++) {
                const int at = tile_at<HD>(c, st * 16 + 8 * g);
                qf[st] = *reinterpret_cast<const bf16x8*>(my_rows + at);
                dof[st] = *reinterpret_cast<const bf16x8*>(my_rows + ROWS + at);
                const bf16x8 of = *reinterpret_cast<const bf16x8*>(my_rows + 2 * ROWS + at);
#pragma unroll
                for (int e = 0; e < 8; e++) dpart += (float)dof[st][e] * (float)of[e];
            }
        } else {
            if (pass == 1) __syncthreads();
            // the first K / V tile travels with the rows of Q, dO and O, not behind the reduction that waits for them
            kv_tile.load_untracked(Kp, a.k_ss, 0, a.S, Ksb, wave, lane);
            kv_tile.load_untracked(Vp, a.k_ss, 0, a.S, Vsb, wave, lane);
#pragma unroll
            for (int st = 0; st < KSTEPS; st++) {
                const int d = st * 16 + 8 * g;
                qf[st] = valid_q ? *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.Q) + qoff + d) : zero8;
                dof[st] = valid_q ? *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.dO) + qoff + d) : zero8;
                const bf16x8 of = valid_q ? *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(a.O) + qoff + d) : zero8;
#pragma unroll
                for (int e = 0; e < 8; e++) dpart += (float)dof[st][e] * (float)of[e];
            }
            lse = valid_q ? a.LSE[stat] : 0.f;
        }
        const float Dq = dpart + __shfl_xor(dpart, 32, 64);
        const float lse2 = valid_q ? lse * kLog2e : INFINITY;
        if (STATS && valid_q && g == 0) {
            a.D[stat] = Dq;
            a.L2[stat] = -lse / a.scale;  // start value of the dK / dV kernel's score accumulators
        }

        f32x16 dq[DT];
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) dq[dt][v] = 0.f;

        const int block_qmax = min(a.S - 1, (qblk * QS + QS - 1) * 32 + 31);
        const int n_kt = a.causal ? block_qmax / BKV + 1 : (a.S + BKV - 1) / BKV;
        const int my_qmax = q0 < a.S ? q0 + 31 : -1;
        // STREAM, first pass: the short block's rows are requested under the second tile (the first one still shares the
        // memory system with every block's start-up), or under the only tile
        const int rows_at = pass == 0 && two ? min(1, n_kt - 1) : -1;

        auto tile = [&](int kt, auto masked_c) {
            constexpr bool MASKED = decltype(masked_c)::value;  // false: no key of the tile is masked for this wave
            const int buf = STREAM ? ((kt + par) & 1) : 0;
            const bf16_t* Ks = Ksb + (ABL == kAblTileLoads ? 0 : (STREAM ? buf : (kt & 1))) * KV;
            const bf16_t* Vs = Vsb + (ABL == kAblTileLoads ? 0 : (STREAM ? buf : (kt & 1))) * KV;
            wait_direct_loads();  // this wave's part of tile kt has landed
            __syncthreads();      // every wave is done with the tile before, whose buffer the next loads overwrite
            if (STREAM) {
                // the next tile of the stream: this pass's, or the first one of the short block
                const bool more = kt + 1 < n_kt;
                if (more || (pass == 0 && two)) {
                    const int first = more ? (kt + 1) * BKV : 0;
                    kv_tile.load_untracked(Kp, a.k_ss, first, a.S, Ksb + (buf ^ 1) * KV, wave, lane);
                    kv_tile.load_untracked(Vp, a.k_ss, first, a.S, Vsb + (buf ^ 1) * KV, wave, lane);
                }
                if (kt == rows_at) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the long block's rows have been read
                    request_rows(qblk_short);
                }
            } else if (ABL != kAblTileLoads && kt + 1 < n_kt) {
                kv_tile.load_untracked(Kp, a.k_ss, (kt + 1) * BKV, a.S, Ksb + ((kt + 1) & 1) * KV, wave, lane);
                kv_tile.load_untracked(Vp, a.k_ss, (kt + 1) * BKV, a.S, Vsb + ((kt + 1) & 1) * KV, wave, lane);
            }
#pragma unroll
            for (int sub = 0; sub < 2; sub++) {
                const int k0 = kt * BKV + sub * 32;
                if (MASKED && (k0 >= a.S || my_qmax < 0 || (a.causal && k0 > my_qmax))) continue;
                f32x16 s, dp;
#pragma unroll
                for (int v = 0; v < 16; v++) { s[v] = 0.f; dp[v] = -Dq; }  // the MFMA chain delivers dP - D
#pragma unroll
                for (int st = 0; st < KSTEPS; st++) {
                    const bf16x8 kf = ABL == kAblOperandReads ? dof[st] : *reinterpret_cast<const bf16x8*>(Ks + tile_at<HD>(sub * 32 + c, st * 16 + 8 * g));
                    const bf16x8 vf = ABL == kAblOperandReads ? qf[st] : *reinterpret_cast<const bf16x8*>(Vs + tile_at<HD>(sub * 32 + c, st * 16 + 8 * g));
                    if (ABL == kAblScoreMfmas) {
                        s[st] += (float)kf[0];
                        dp[st] += (float)vf[0];
                    } else {
                        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[st], s, 0, 0, 0);
                        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, dof[st], dp, 0, 0, 0);
                    }
                }
                bf16x8 dsf[2];
                // a query past the end has LSE = +inf; keys past the end (their tile rows repeat the last
                // key) and keys above the causal diagonal are masked
                float p[16];
#pragma unroll
                for (int v = 0; v < 16; v++) p[v] = ABL == kAblSoftmax ? s[v] : fast_exp2(fmaf(s[v], a.scale_log2e, -lse2));
                if (MASKED && ((a.causal && k0 + 31 > q0) || k0 + 32 > a.S)) {
                    const int rel = min(a.causal ? q : a.S - 1, a.S - 1) - k0;  // keys k0 + row > rel are masked
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        if (acc_row(v, g) > rel) p[v] = 0.f;
                }
#pragma unroll
                for (int v = 0; v < 16; v++) dsf[v >> 3][v & 7] = (bf16_t)(ABL == kAblSoftmax ? dp[v] : p[v] * dp[v]);
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const bf16x8 ktr = ABL == kAblTransposedReads ? qf[dt * 2 + t] : lds_tr_operand_swz<HD>(Ks, sub * 32, dt * 32, t, lane);
                        if (ABL == kAblSecondMfmas) dq[dt][0] += (float)ktr[0] * (float)dsf[t][0];
                        else dq[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktr, dsf[t], dq[dt], 0, 0, 0);
                    }
            }
        };
        const int n_plain = my_qmax < 0 ? 0 : min(n_kt, min(a.causal ? (q0 + 1) / BKV : n_kt, a.S / BKV));
        int kt = 0;
        attn_stamp<TL>(a, 1, kStampLoop + kStampsPerPass * pass, lane, wave);
        for (; kt < n_plain; kt++) tile(kt, std::false_type{});
        for (; kt < n_kt; kt++) tile(kt, std::true_type{});
        attn_stamp<TL>(a, 1, kStampLoopEnd + kStampsPerPass * pass, lane, wave);
        par = (par + n_kt) & 1;
        if (valid_q) {
            bf16_t* dQp = static_cast<bf16_t*>(a.dQ) + qoff;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int vg = 0; vg < 4; vg++) {
                    if (dt * 32 + 8 * vg >= HD) continue;
                    float x[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] = dq[dt][vg * 4 + e] * a.scale;
                    if (a.rope) unrotate_pairs<2>(x, a.rope + (size_t)q * (HD / 2) + (dt * 32 + 8 * vg + 4 * g) / 2);
                    bf16x4 w;
#pragma unroll
                    for (int e = 0; e < 4; e++) w[e] = (bf16_t)x[e];
                    *reinterpret_cast<bf16x4*>(dQp + dt * 32 + 8 * vg + 4 * g) = w;
                }
        }
        attn_stamp<TL>(a, 1, kStampStored + kStampsPerPass * pass, lane, wave);
    }
}

}  // namespace

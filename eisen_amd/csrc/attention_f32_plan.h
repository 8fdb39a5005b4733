// How the launches of f32 attention on the matrix cores (attention_f32.hip) are laid out: waves per workgroup, grids, LDS.
#pragma once
#include <algorithm>
#include <cstddef>

// Waves of a workgroup, at most: two to a SIMD where their registers allow it (head sizes up to 32; k8: the head size rounded up to 8 * k8).  Eight
// instead of four, forward / dQ pass of the backward in us, causal: 1 x 2000, 2 heads of 32 24.4 / 23.5 and 57.5 / 45.7; 1 x 4000, one head 44.4 / 42.1 and
// 106 / 82; 1 x 448, 3 heads 8.8 / 9.2 and 19.5 / 17.2.
constexpr int f32_attn_max_waves(int k8) { return k8 <= 4 ? 8 : 4; }

// Where the waves of a workgroup meet, in floats: nothing for one wave, as large grids have it.  (Held for eight or four waves whatever the launch had, a
// workgroup of one wave took 32 to 64 KB, and two to five were on a CU where registers allow four to twelve: 16 x 512, 8 heads of 128, backward 624 us, now 383,
// forward 128 / 93; 32 x 256, 8 of 32 98 / 51 and 24.3 / 19.5; 256 x 16, 8 of 16 31.7 / 13.8 and 10.1 / 6.2.)
constexpr int kF32AttnTile = 16 * 64;  // a wave's 32 x 32 results
constexpr int f32_attn_fwd_meet(int dt, int waves) { return (waves - 1) * (dt * kF32AttnTile + 128); }
constexpr int f32_attn_dq_meet(int dt, int waves) { return (waves - 1) * dt * kF32AttnTile; }
constexpr int f32_attn_dkv_meet(int waves) { return waves > 1 ? 2 * waves * kF32AttnTile : 0; }

// Enough waves for two per SIMD of the chip, but none without at least one tile of the longest row.
inline int f32_attn_waves(long long blocks, int tiles, int most) {
    int w = 1;
    while (w < most && blocks * w < 2048 && 2 * w <= tiles) w *= 2;
    return w;
}

// One launch for the backward, or one for dQ and one for dK and dV.  One lets either pass fill the gaps of the other and has a dK/dV item read the rows of O as well;
// for head sizes above 96, whose one wave per SIMD waits for all of an item's rows, that costs more than it gives once each pass fills the chip by itself.
// Two / one, us, causal, batch x sequence, query heads on KV heads, head size: 16 x 256 8 on 8 128 128 / 140; 8 x 512 8 on 8 128 192 / 209; 16 x 512 8 on 8 128
// 331 / 382; 16 x 512 16 on 4 128 663 / 747; 64 x 128 8 on 8 128 156 / 171; 128 x 32 8 on 8 128 49 / 53; 8 x 512 16 on 8 100 504 / 556; 512 x 32 8 on 8 100 297 / 307.
// Below 1024 key blocks it depends on the shape: 4 x 512 8 on 8 128 131 / 137; 2 x 1500 8 on 4 128 407 / 423; but 4 x 512 16 on 4 128 247 / 215; 80 x 64 16 on 4 128
// 153 / 145; 1 x 800 8 on 8 128 134 / 92.  Smaller heads: 32 x 256 8 on 8 32 64 / 51; 16 x 512 8 on 8 64 165 / 172; 8 x 512 8 on 2 64 131 / 103; 2 x 2000 8 on 2 96
// 686 / 591; 16 x 512 8 on 8 96 254 / 273; 512 x 32 8 on 8 96 156 / 153.  And two where the workgroups of one have more threads than a launch takes.
struct F32AttnPlan {
    long long qblocks, kblocks, dq_groups;  // dq_groups: workgroups of the combined backward that form dQ, of wk / wq query blocks each
    int wq, wk;
    bool one;  // the backward is one launch
    size_t fwd_lds, dq_lds, dkv_lds, bwd_lds;  // bytes
};
inline F32AttnPlan f32_attn_plan(int k8, int B, int S, int Hq, int Hkv) {
    const int n_t = (S + 31) / 32, dt = (k8 + 3) / 4, most = f32_attn_max_waves(k8);
    F32AttnPlan p{};
    p.qblocks = (long long)n_t * Hq * B;
    p.kblocks = (long long)n_t * Hkv * B;
    p.wq = f32_attn_waves(p.qblocks, n_t, most);
    p.wk = f32_attn_waves(p.kblocks, n_t * (Hq / Hkv), most);
    const int together = p.wk / p.wq;  // (wq <= wk: there are no fewer query blocks than key blocks)
    p.dq_groups = (p.qblocks + together - 1) / together;
    p.fwd_lds = f32_attn_fwd_meet(dt, p.wq) * sizeof(float);
    p.dq_lds = f32_attn_dq_meet(dt, p.wq) * sizeof(float);
    p.dkv_lds = f32_attn_dkv_meet(p.wk) * sizeof(float);
    p.bwd_lds = std::max(together * p.dq_lds, p.dkv_lds);
    p.one = !(k8 > 12 && p.kblocks >= 1024) && (p.kblocks + p.dq_groups) * 64 * p.wk < (1ll << 32);
    return p;
}

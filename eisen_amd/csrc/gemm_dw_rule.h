// Whether the weight gradients of several layers over K tokens are formed by the launch for many layers (gemm_dw.hip, gemm_f32_sliced.hip) or by a launch each.
#pragma once
#include <algorithm>
#include <cstddef>

// That launch gives a workgroup a tile's whole contraction; a launch each may split it.  So few tiles over many tokens wait for one workgroup, about 4 + K / 450 us in bf16 and
// 5 + K / 80 in f32 (tiles of 32 x 32, for fewer than 64 tiles of 64 x 64 over 1024 tokens or more: 5 + K / 170), more than 256 tiles in proportion; a launch each takes about
// 7 us and what its tiles need.  Sets, a launch each / one launch, us: bf16 1 of 512 x 512 over 2048 10 / 10, 4096 12 / 19, 8192 15 / 34; 2 of 64 x 64 over 4096 17 / 14, 8192 16 / 22;
// 3 of 256 x 256 over 4096 25 / 15, 8192 31 / 28, 16384 38 / 53; 1 of 1024 x 1024 over 4096 25 / 18, 16384 66 / 58; the ~14 M model's 7 of one layer over 8192 80 / 33.  f32 1 of
// 512 x 512 over 1024 10 / 19, 2 over 1024 19 / 20, 4 over 4096 86 / 62; 2 of 64 x 64 over 1024 16 / 11, 2048 16 / 17, 4096 17 / 29; the ~14 M model's layer over 4096 107 / 63.
// (Every set measured, 13 of one to 14 products over 512 to 16384 tokens, goes where it is faster, or within 2 us.)
inline bool eisen_dw_together(bool bf16, size_t n, const size_t* M, const size_t* N, size_t K) {
    double tiles = 0.0;
    for (size_t p = 0; p < n; p++) tiles += (double)((M[p] + 63) / 64) * (double)((N[p] + 63) / 64);
    const double k = (double)K, rounds = std::max(1.0, tiles / 256.0);
    const double each = 7.0 * (double)n + tiles * k / (bf16 ? 65536.0 : 20000.0);
    const double together = bf16 ? 4.0 + k / 450.0 * rounds : 5.0 + k / (tiles < 64.0 && K >= 1024 ? 170.0 : 80.0) * rounds;
    return together <= each;
}

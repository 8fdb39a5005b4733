// Whether the weight gradients of several layers over K tokens are formed by the launch for many layers (gemm_dw.hip, gemm_f32_sliced.hip) or by a launch each.
#pragma once
#include <algorithm>
#include <cstddef>

// That launch gives a workgroup a tile's whole contraction; a launch each may split it.  So few tiles over many tokens wait for one workgroup, about 4 + K / 360 us in bf16 and
// 5 + K / 80 in f32 (tiles of 32 x 32, for fewer than 64 tiles of 64 x 64 over 1024 tokens or more: 5 + K / 170), more than 256 tiles in proportion; a launch each takes about
// 7 us and what its tiles need.  Sets, a launch each / one launch, us: bf16 2 of 64 x 64 over 4096 14 / 15, 8192 14 / 25; 2 of 288 x 768 over 4096 23 / 19, 8192 28 / 36, 16384 41 / 70;
// 3 of 256 x 256 over 4096 23 / 15, 8192 30 / 27; 2 of 512 x 1024 over 2048 23 / 11; 2 of 1024 x 1024 over 4096 54 / 30; the ~14 M model's 7 of one layer over 8192 80 / 33.  f32 2 of
// 512 x 512 over 1024 19 / 20, 4 over 4096 86 / 62; 2 of 64 x 64 over 1024 16 / 11, 2048 16 / 17, 4096 17 / 29; the ~14 M model's layer over 4096 107 / 63.
// (Of 700 sets of 2 to 8 equal products of 64 x 64 to 2048 x 1792 over 64 to 16384 tokens the rule's choice costs a tenth or more with 14, most of them pairs over 16384, and 28 % at most.)
inline bool eisen_dw_together(bool bf16, size_t n, const size_t* M, const size_t* N, size_t K) {
    double tiles = 0.0;
    for (size_t p = 0; p < n; p++) tiles += (double)((M[p] + 63) / 64) * (double)((N[p] + 63) / 64);
    const double k = (double)K, rounds = std::max(1.0, tiles / 256.0);
    const double each = 7.0 * (double)n + tiles * k / (bf16 ? 65536.0 : 20000.0);
    const double together = bf16 ? 4.2 + k / 360.0 * rounds : 5.0 + k / (tiles < 64.0 && K >= 1024 ? 170.0 : 80.0) * rounds;
    return together <= each;
}

// Whether that launch is better for one product alone: hardly ever.  Its own / that launch, us: bf16 64 x 64 x 64 3.2 / 4.5, x 1024 4.3 / 6.9, 256 x 256 x 512 4.1 / 5.9, 768 x 768 x 4096 17 / 18,
// 1536 x 1536 x 4096 36 / 54; f32 64 x 64 x 64 4.0 / 6.4, 256 x 1024 x 1024 8.8 / 18.5, 1024 x 1024 x 4096 53 / 59.  But where its tiles are one or two whole rounds of the chip and a launch of its
// own splits: bf16 1024 x 1024 x 4096 26 / 18, 1024 x 2048 x 2048 28 / 20, 256 x 8192 x 4096 38 / 29.
inline bool eisen_dw_alone(bool bf16, size_t M, size_t N, size_t K) {
    const size_t tiles = M / 64 * (N / 64);
    return bf16 && K >= 2048 && M % 64 == 0 && N % 64 == 0 && (tiles == 256 || tiles == 512);
}

// The same for the bf16 products of one node (a weight, or the weights that share an input), whose launch each is one launch too, and which are not left for others: where weight
// gradients keep to the tape.  (By this, the bits of narrow layers over few tokens are those of a pass's launch.)
// Steps kept to the tape with bf16 nodes by this and f32 ones by their own launches / all nodes by eisen_dw_together, a launch per product where it says no, us: the ~14 M model 1606 / 1875, in
// f32 2737 / 2954; hidden 1536, 3 layers, 4096 tokens 3723 / 3773; hidden 1024, 4 layers, 1024 tokens 1409 / 1425; hidden 128 in f32, 4 layers, 512 tokens 625 / 682.
inline bool eisen_dw_node(size_t n, const size_t* M, const size_t* N, size_t K) {
    double tiles = 0.0;
    for (size_t p = 0; p < n; p++) tiles += (double)((M[p] + 63) / 64) * (double)((N[p] + 63) / 64);
    if (n == 1 && tiles >= 256.0) return eisen_dw_alone(true, M[0], N[0], K);
    return 4.2 + (double)K / 360.0 * std::max(1.0, tiles / 256.0) <= 7.0 + tiles * (double)K / 65536.0;
}

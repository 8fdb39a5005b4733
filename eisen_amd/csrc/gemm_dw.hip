// Weight gradients of many Linear layers in one launch: C_p (+)= A_p^T B_p with bf16 A_p [K][M_p], B_p [K][N_p] and f32 C_p, for the layers of
// a backward pass, whose products share the contraction (the tokens of the pass) and little else.
//
// What bounds it: the LDS pipe.  Both operands are stored along their rows, so an MFMA operand of 32 x 16 is two transposing reads of 8 clocks each
// and its share of the direct loads' writes.  So the four waves of a workgroup do not share a tile's operands but its contraction: a wave owns the whole tile
// for every fourth 16-deep slice, through a private ring of four with no barrier, and the four sums meet in LDS once, added in wave order.  A tile of 128 x 64 reads 6
// operands per 8 MFMAs, one of 64 x 64 8; but the former leaves one workgroup on a CU, whose start and end nothing hides.  Both give the same bits: the slices of a wave do not
// depend on the tile.
// The sums of a few slices are added up apart, so that no accumulator rounds a long one, nor the total many short ones (`run`).  Products of fewer than 64 tiles of 64 x 64 over
// more than 2048 tokens, which a launch of their own splits, come in parts of 4096 tokens, each added to C before the next, and add the waves' sums two and two (`dw_exact`).
// Error against float64, these / all of a wave's slices in one accumulator / a launch of its own: 256 x 1024 x 2048 8.1e-8 / 1.3e-7 / 8.6e-8, x 4096 9.2e-8 / 1.9e-7 / 9.2e-8, x
// 8192 1.1e-7 / 2.7e-7 / 1.1e-7, x 16384 1.2e-7 / 4.0e-7 / 1.4e-7; 8192 x 256 x 8192 1.1e-7 / 2.7e-7 / 4.0e-7; 1024 x 1024 x 4096 9.2e-8 / 1.9e-7 / 2.7e-7; 288 x 768 x
// 1351 7.7e-8 / 1.1e-7 / 9.1e-8; of positive operands 256 x 1024 x 8192 4.7e-8 / 1.3e-7 / 4.7e-8.  Few tiles, these / in one part / a launch of its own: 256 x 256 x 4096 9.1e-8 / 9.3e-8 /
// 9.2e-8, x 8192 9.5e-8 / 1.10e-7 / 1.00e-7, x 16384 1.00e-7 / 1.22e-7 / 1.12e-7, 64 x 64 x 8192 9.5e-8 / 1.10e-7 / 9.9e-8.
// Rates: 4 x 1536 x 1024 over 8192 tokens 710 TFLOP/s, 12 x 1024 x 1024 over 4096 630.  A pass's layers, a launch each / this, us:
// hidden 256, ffn 1024, 6 layers and a head of 8192 over 8192 tokens 636 / 268 (254 without the parts); 288, 768, 4 layers over 1351 187 / 33; 512, 1536, 4 layers over 4096 460 / 226;
// 720, 2120, 6 layers over 896 456 / 241.
// (Tried: wave tiles of 128 x 128, which leave no registers for sums apart, 209 us for the first of these sets and the error in the middle above; with them a persistent grid that
// requests the next tile's slices before the meeting, 258 -> 285 us at 8192 x 8192 x 1024, and a meeting in which a wave receives only the quarter that it stores, 258 -> 289.
// Compensated sums instead of plain ones: 180 registers in scratch, or 5 to 20 % longer with 64 x 64; a carry from each run into the next for the few tiles' products alone, a loop of its
// own, 276 instead of 268 for the first of these sets.)
//
// Operand rows start on 16-byte boundaries and sides are multiples of 8.  Columns past the end re-read the last chunk and reach only outputs that are not
// stored; contraction indices past the end re-read the last one, and both operands are zeroed there.
#include "gemm_common.cuh"

namespace {

constexpr int kCols = 64, kSlice = 16, kRing = 4, kWaves = 4, kPart = 4096;

__host__ __device__ constexpr bool dw_exact(int M, int N, int K) { return K > 2048 && ((M + 63) / 64) * ((N + 63) / 64) < 64; }

template <int ROWS>
using DwStages = bf16_t[kWaves][kRing][DirectOperandTile<ROWS, false, kSlice, 1>::ELEMS + DirectOperandTile<kCols, false, kSlice, 1>::ELEMS];

// A tile's sum over the K tokens from k0 on, by the whole workgroup; added to C where add_old.  pairs: the waves' sums are added two and two.
template <int ROWS>
__device__ __forceinline__ void dw_tile(const DwProduct& pr, DwStages<ROWS>& lds, int m0, int n0, int k0, int K, bool add_old, bool pairs) {
    using TA = DirectOperandTile<ROWS, false, kSlice, 1>;
    using TB = DirectOperandTile<kCols, false, kSlice, 1>;
    constexpr int TM = ROWS / 32, TN = kCols / 32, LOADS = TA::LOADS + TB::LOADS, STAGE = TA::ELEMS + TB::ELEMS;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = pr.M, N = pr.N;
    const int slices = (K + kSlice - 1) / kSlice, n_mine = slices > wave ? (slices - wave + kWaves - 1) / kWaves : 0, n_parts = min(kWaves, slices);
    const char* A = static_cast<const char*>(pr.A) + ((long long)(k0 + wave * kSlice) * M + m0) * 2;
    const char* B = static_cast<const char*>(pr.B) + ((long long)(k0 + wave * kSlice) * N + n0) * 2;
    const int a_last = (M - 1 - m0) / 8, b_last = (N - 1 - n0) / 8;
    unsigned a_off[TA::LOADS], b_off[TB::LOADS];  // a lane's bytes in a slice
#pragma unroll
    for (int i = 0; i < TA::LOADS; i++) {
        int row, chunk;
        TA::lane_chunk(i, 0, lane, row, chunk);
        a_off[i] = (unsigned)(row * M + min(chunk, a_last) * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < TB::LOADS; i++) {
        int row, chunk;
        TB::lane_chunk(i, 0, lane, row, chunk);
        b_off[i] = (unsigned)(row * N + min(chunk, b_last) * 8) * 2u;
    }
    const unsigned lds0 = (unsigned)(size_t)(lds_void_ptr)(&lds[wave][0][0]);
    const int tail = K - (slices - 1) * kSlice;  // rows of the last slice
    const bool tail_mine = tail < kSlice && (slices - 1) % kWaves == wave;
    int to_issue = n_mine;  // slices not yet requested
    auto load = [&](auto stage_c, auto h_c) __attribute__((always_inline)) {
        constexpr int st = decltype(stage_c)::value, h = decltype(h_c)::value;
        if constexpr (h < TA::LOADS) load_to_lds_16_at<st * STAGE * 2 + h * 1024>(A, a_off[h], lds0);
        else load_to_lds_16_at<(st * STAGE + TA::ELEMS) * 2 + (h - TA::LOADS) * 1024>(B, b_off[h - TA::LOADS], lds0);
    };
    auto cut_last = [&]() __attribute__((always_inline)) {  // if the next slice is the contraction's last, rows past the end re-read the last one
        if (tail_mine && to_issue == 1) {
#pragma unroll
            for (int i = 0; i < TA::LOADS; i++) a_off[i] -= (unsigned)max(i * TA::RPB + lane / TA::CPR - (tail - 1), 0) * (unsigned)M * 2u;
#pragma unroll
            for (int i = 0; i < TB::LOADS; i++) b_off[i] -= (unsigned)max(i * TB::RPB + lane / TB::CPR - (tail - 1), 0) * (unsigned)N * 2u;
        }
    };
    auto advance = [&]() __attribute__((always_inline)) {  // (behind a wave's last slice its loads are repeated, into stages that nobody reads)
        to_issue--;
        if (to_issue > 0) {
            A += (unsigned)M * (kWaves * kSlice * 2);
            B += (unsigned)N * (kWaves * kSlice * 2);
            cut_last();
        }
    };

    f32x16 acc[TM][TN] = {}, total[TM][TN] = {};
    const int run = K <= 2048 ? 4 : K <= 6144 ? 8 : 16;  // slices whose sum is added to the total, a multiple of kRing
    auto add_to_total = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < TM; x++)
#pragma unroll
            for (int y = 0; y < TN; y++) {
                total[x][y] += acc[x][y];
                acc[x][y] = f32x16{};
            }
    };
    bf16x8 a[2][TM], b[2][TN];
    auto read_frag = [&](auto buf_c, auto stage_c, auto q_c) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_c)::value, st = decltype(stage_c)::value, q = decltype(q_c)::value;
        const bf16_t* As = lds[wave][st];
        const bf16_t* Bs = As + TA::ELEMS;
        if constexpr (q == 0) a[buf][0] = TA::fragment(As, 0, 0, lane);
        else if constexpr (q <= TN) b[buf][q - 1] = TB::fragment(Bs, (q - 1) * 32, 0, lane);
        else a[buf][q - TN] = TA::fragment(As, (q - TN) * 32, 0, lane);
    };
    auto step = [&](auto stage_c, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(stage_c)::value, cur = ST & 1, next = (ST + 1) % kRing;
        using NC = std::integral_constant<int, next>;
        using BC = std::integral_constant<int, cur ^ 1>;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (tail_mine && i == n_mine - 1) {
            const int k = 8 * (lane >> 5);
#pragma unroll
            for (int h = 0; h < TM; h++) a[cur][h] = zero_from(a[cur][h], k, tail);
#pragma unroll
            for (int h = 0; h < TN; h++) b[cur][h] = zero_from(b[cur][h], k, tail);
        }
        wait_loads_but<(kRing - 2) * LOADS>();
        __builtin_amdgcn_sched_barrier(0);
        static_for<TM * TN>([&](auto m_c) {
            constexpr int mi = decltype(m_c)::value, x = mi / TN, y = mi % TN;
            acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[cur][x], b[cur][y], acc[x][y], 0, 0, 0);
            if constexpr (mi < TM + TN) read_frag(BC{}, NC{}, m_c);
            if constexpr (mi < LOADS) load(stage_c, m_c);
            __builtin_amdgcn_sched_barrier(0);
        });
        advance();
    };

    if (n_mine > 0) {
        cut_last();
        static_for<kRing>([&](auto s_c) {
            static_for<LOADS>([&](auto h_c) { load(s_c, h_c); });
            advance();
        });
        wait_loads_but<(kRing - 1) * LOADS>();
        static_for<TM + TN>([&](auto q_c) { read_frag(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, q_c); });
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < n_mine; i += kRing) {
            if (i > 0 && i % run == 0) add_to_total();
            static_for<kRing>([&](auto s_c) {
                if (i + decltype(s_c)::value < n_mine) step(s_c, i + decltype(s_c)::value);
            });
        }
        wait_loads_but<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        add_to_total();
    }
    // (a wave's partial sums take the place of its own slices)
    float* mine = reinterpret_cast<float*>(&lds[wave][0][0]);
    auto place = [](int r, int n) { return r * kCols + (n ^ ((r >> 2 & 1) * 32)); };
    static_assert(sizeof(lds[0]) >= 64 * kCols * sizeof(float), "64 rows of partial sums");
#pragma unroll
    for (int half = 0; half < ROWS / 64; half++) {
        if (half > 0) __syncthreads();
        if (n_mine > 0) {
            const int c = lane & 31, gh = lane >> 5;
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) mine[place(i * 32 + 8 * (v / 4) + 4 * gh + (v % 4), j * 32 + c)] = total[2 * half + i][j][v];
        }
        __syncthreads();
        for (int idx = tid; idx < 64 * kCols / 8; idx += 64 * kWaves) {
            const int r = idx / (kCols / 8), cg = idx % (kCols / 8), m = m0 + half * 64 + r, n = n0 + cg * 8;
            if (m >= M || n >= N) continue;
            float* dst = static_cast<float*>(pr.C) + (long long)m * N + n;
            float val[8] = {};
            const float* src = reinterpret_cast<const float*>(&lds[0][0][0]) + place(r, cg * 8);
            float held[8] = {};
            for (int w = 0; w < n_parts; w++) {
                if (pairs && w == 2) {
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        held[e] = val[e];
                        val[e] = 0.f;
                    }
                }
                const float4 lo = *reinterpret_cast<const float4*>(src + w * (kRing * STAGE / 2)), hi = *reinterpret_cast<const float4*>(src + w * (kRing * STAGE / 2) + 4);
                val[0] += lo.x; val[1] += lo.y; val[2] += lo.z; val[3] += lo.w;
                val[4] += hi.x; val[5] += hi.y; val[6] += hi.z; val[7] += hi.w;
            }
            if (pairs) {
#pragma unroll
                for (int e = 0; e < 8; e++) val[e] += held[e];
            }
            float4 lo = make_float4(val[0], val[1], val[2], val[3]), hi = make_float4(val[4], val[5], val[6], val[7]);
            if (add_old) {
                const float4 o0 = reinterpret_cast<const float4*>(dst)[0], o1 = reinterpret_cast<const float4*>(dst)[1];
                lo.x += o0.x; lo.y += o0.y; lo.z += o0.z; lo.w += o0.w;
                hi.x += o1.x; hi.y += o1.y; hi.z += o1.z; hi.w += o1.w;
            }
            reinterpret_cast<float4*>(dst)[0] = lo;
            reinterpret_cast<float4*>(dst)[1] = hi;
        }
    }
}

template <int ROWS, bool EXACT>
__global__ __launch_bounds__(64 * kWaves, ROWS == 64 ? 2 : 1) void gemm_dw_kernel(DwArgs g) {
    __shared__ __attribute__((aligned(1024))) DwStages<ROWS> lds;
    const int lane = threadIdx.x & 63;

    // which product this tile belongs to: every lane looks at one
    int t = xcd_contiguous_id(blockIdx.x, g.tiles);
    const int p = __popcll(__ballot(lane < g.n && t >= g.tile_end[lane]));
    const DwProduct& pr = g.p[p];
    if (p > 0) t -= g.tile_end[p - 1];
    const int M = pr.M, N = pr.N, K = g.K;
    int mt, nt;
    block_tile<4, 8>(t, (M + ROWS - 1) / ROWS, (N + kCols - 1) / kCols, mt, nt);
    const int m0 = __builtin_amdgcn_readfirstlane(mt * ROWS), n0 = __builtin_amdgcn_readfirstlane(nt * kCols);

    if constexpr (EXACT) {
        const bool exact = dw_exact(M, N, K);
        const int part = exact ? min(K, kPart) : K;
        for (int k0 = 0; k0 < K; k0 += part) {
            if (k0 > 0) __syncthreads();  // the last part's sums have been read
            dw_tile<ROWS>(pr, lds, m0, n0, k0, min(part, K - k0), k0 > 0 || pr.accumulate, exact);
        }
    } else {
        dw_tile<ROWS>(pr, lds, m0, n0, 0, K, pr.accumulate, false);
    }
}

}  // namespace

void eisen_gemm_launch_dw(eisen_ctx* ctx, const DwArgs& g, int rows) {
    bool exact = false;
    for (int p = 0; p < g.n; p++) exact = exact || dw_exact(g.p[p].M, g.p[p].N, g.K);
    auto launch = [&](auto rows_c) {
        constexpr int ROWS = decltype(rows_c)::value;
        if (exact) gemm_dw_kernel<ROWS, true><<<(unsigned)g.tiles, 64 * kWaves, 0, ctx->stream>>>(g);
        else gemm_dw_kernel<ROWS, false><<<(unsigned)g.tiles, 64 * kWaves, 0, ctx->stream>>>(g);
    };
    if (rows == 128) launch(std::integral_constant<int, 128>{});
    else launch(std::integral_constant<int, 64>{});
}

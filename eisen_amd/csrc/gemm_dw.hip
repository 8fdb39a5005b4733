// Weight gradients of many Linear layers in one launch: C_p (+)= A_p^T B_p with bf16 A_p [K][M_p], B_p [K][N_p] and f32 C_p, for the layers of
// a backward pass, whose products share the contraction (the tokens of the pass) and little else.
//
// What bounds it: the LDS pipe.  Both operands are stored along their rows, so an MFMA operand of 32 x 16 is two transposing reads of 8 clocks each
// and its share of the direct loads' writes.  A wave that owns a whole 128 x 128 tile reads 8 operands per 16 MFMAs, 12 clocks of LDS per contraction index and tile where
// the matrix pipes need 8 (measured 13); 64 x 64 tiles take twice that for the same outputs, tiles shared by four waves of 64 x 64 20.  So the four waves of a workgroup do not share a tile's operands but its
// contraction: a wave takes every fourth 16-deep slice through a private ring of four, with no barrier, and the four sums meet in LDS once, added in
// wave order.  The accumulators of a 128 x 128 wave tile leave one workgroup on a CU, whose start and end (7 us of the 13 that a tile takes over 1024 tokens)
// nothing hides; tiles of 64 run two.  Both give the same bits: the slices of a wave do not depend on the tile.
// Rates: 12 x 1024 x 1024 over 4096 tokens 890 TFLOP/s, 2048 x 2048 over 8192 1070 with operands in the caches.  A pass's layers, a launch each / this, us:
// hidden 256, ffn 1024, 6 layers and a head of 8192 over 8192 tokens 626 / 209; 288, 768, 4 layers over 1351 186 / 33; 512, 1536, 4 layers over 4096 423 / 137;
// 720, 2120, 6 layers over 896 403 / 174.
// (Tried: a persistent grid that requests the next tile's slices before the meeting, 258 -> 285 us at 8192 x 8192 x 1024; a meeting in which a wave receives only
// the quarter that it stores, 258 -> 289; rings of two with four 64 x 64 workgroups per CU, equal or slower from 800 tokens on.)
//
// Operand rows start on 16-byte boundaries and sides are multiples of 8.  Columns past the end re-read the last chunk and reach only outputs that are not
// stored; contraction indices past the end re-read the last one, and both operands are zeroed there.
#include "gemm_common.cuh"

namespace {

constexpr int kSlice = 16, kRing = 4, kWaves = 4;

template <int TILE>
__global__ __launch_bounds__(64 * kWaves) void gemm_dw_kernel(DwArgs g) {
    using T = DirectOperandTile<TILE, false, kSlice, 1>;
    constexpr int TM = TILE / 32, LOADS = T::LOADS, STAGE = 2 * T::ELEMS;
    __shared__ __attribute__((aligned(1024))) bf16_t lds[kWaves][kRing][STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // which product this tile belongs to: every lane looks at one
    int t = xcd_contiguous_id(blockIdx.x, g.tiles);
    const int p = __popcll(__ballot(lane < g.n && t >= g.tile_end[lane]));
    const DwProduct& pr = g.p[p];
    if (p > 0) t -= g.tile_end[p - 1];
    const int M = pr.M, N = pr.N, K = g.K;
    int mt, nt;
    block_tile<4, 8>(t, (M + TILE - 1) / TILE, (N + TILE - 1) / TILE, mt, nt);
    const int m0 = __builtin_amdgcn_readfirstlane(mt * TILE), n0 = __builtin_amdgcn_readfirstlane(nt * TILE);

    const int slices = (K + kSlice - 1) / kSlice, n_mine = slices > wave ? (slices - wave + kWaves - 1) / kWaves : 0, n_parts = min(kWaves, slices);
    const char* A = static_cast<const char*>(pr.A) + ((long long)wave * kSlice * M + m0) * 2;
    const char* B = static_cast<const char*>(pr.B) + ((long long)wave * kSlice * N + n0) * 2;
    const int a_last = (M - 1 - m0) / 8, b_last = (N - 1 - n0) / 8;
    unsigned a_off[LOADS], b_off[LOADS];  // a lane's bytes in a slice
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        int row, chunk;
        T::lane_chunk(i, 0, lane, row, chunk);
        a_off[i] = (unsigned)(row * M + min(chunk, a_last) * 8) * 2u;
        b_off[i] = (unsigned)(row * N + min(chunk, b_last) * 8) * 2u;
    }
    const unsigned lds0 = (unsigned)(size_t)(lds_void_ptr)(&lds[wave][0][0]);
    const int tail = K - (slices - 1) * kSlice;  // rows of the last slice
    const bool tail_mine = tail < kSlice && (slices - 1) % kWaves == wave;
    int to_issue = n_mine;  // slices not yet requested
    auto load = [&](auto stage_c, auto h_c) __attribute__((always_inline)) {
        constexpr int st = decltype(stage_c)::value, h = decltype(h_c)::value, i = h % LOADS;
        load_to_lds_16_at<st * STAGE * 2 + (h < LOADS ? 0 : T::ELEMS * 2) + i * 1024>(h < LOADS ? A : B, h < LOADS ? a_off[i] : b_off[i], lds0);
    };
    auto cut_last = [&]() __attribute__((always_inline)) {  // if the next slice is the contraction's last, rows past the end re-read the last one
        if (tail_mine && to_issue == 1) {
#pragma unroll
            for (int i = 0; i < LOADS; i++) {
                const unsigned past = (unsigned)max(i * T::RPB + lane / T::CPR - (tail - 1), 0);
                a_off[i] -= past * (unsigned)M * 2u;
                b_off[i] -= past * (unsigned)N * 2u;
            }
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

    f32x16 acc[TM][TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
    bf16x8 a[2][TM], b[2][TM];
    auto read_frag = [&](auto buf_c, auto stage_c, auto q_c) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_c)::value, st = decltype(stage_c)::value, q = decltype(q_c)::value;
        const bf16_t* As = lds[wave][st];
        const bf16_t* Bs = As + T::ELEMS;
        if constexpr (q == 0) a[buf][0] = T::fragment(As, 0, 0, lane);
        else if constexpr (q <= TM) b[buf][q - 1] = T::fragment(Bs, (q - 1) * 32, 0, lane);
        else a[buf][q - TM] = T::fragment(As, (q - TM) * 32, 0, lane);
    };
    auto step = [&](auto stage_c, int i) __attribute__((always_inline)) {
        constexpr int ST = decltype(stage_c)::value, cur = ST & 1, next = (ST + 1) % kRing;
        using NC = std::integral_constant<int, next>;
        using BC = std::integral_constant<int, cur ^ 1>;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (tail_mine && i == n_mine - 1) {
            const int k = 8 * (lane >> 5);
#pragma unroll
            for (int h = 0; h < TM; h++) {
                a[cur][h] = zero_from(a[cur][h], k, tail);
                b[cur][h] = zero_from(b[cur][h], k, tail);
            }
        }
        wait_loads_but<(kRing - 2) * 2 * LOADS>();
        __builtin_amdgcn_sched_barrier(0);
        static_for<TM * TM>([&](auto m_c) {
            constexpr int mi = decltype(m_c)::value, x = mi / TM, y = mi % TM;
            acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[cur][x], b[cur][y], acc[x][y], 0, 0, 0);
            if constexpr (TM == 4) {
                if constexpr (mi < 8) read_frag(BC{}, NC{}, m_c);
                else load(stage_c, std::integral_constant<int, mi - 8>{});
            } else {
                read_frag(BC{}, NC{}, m_c);
                load(stage_c, m_c);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        advance();
    };

    if (n_mine > 0) {
        cut_last();
        static_for<kRing>([&](auto s_c) {
            static_for<2 * LOADS>([&](auto h_c) { load(s_c, h_c); });
            advance();
        });
        wait_loads_but<(kRing - 1) * 2 * LOADS>();
        static_for<2 * TM>([&](auto q_c) { read_frag(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, q_c); });
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < n_mine; i += kRing) {
            static_for<kRing>([&](auto s_c) {
                if (i + decltype(s_c)::value < n_mine) step(s_c, i + decltype(s_c)::value);
            });
        }
        wait_loads_but<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // (a wave's partial sums take the place of its own slices)
    float* mine = reinterpret_cast<float*>(&lds[wave][0][0]);
    auto place = [](int r, int n) { return r * TILE + (n ^ ((r >> 2 & 1) * 32)); };
    constexpr int ROWS = 64;
    static_assert(sizeof(lds[0]) >= ROWS * TILE * sizeof(float), "a pass's rows of partial sums");
#pragma unroll
    for (int half = 0; half < TILE / ROWS; half++) {
        if (half > 0) __syncthreads();
        if (n_mine > 0) {
            const int c = lane & 31, gh = lane >> 5;
#pragma unroll
            for (int i = 0; i < ROWS / 32; i++)
#pragma unroll
                for (int j = 0; j < TM; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) mine[place(i * 32 + 8 * (v / 4) + 4 * gh + (v % 4), j * 32 + c)] = acc[ROWS / 32 * half + i][j][v];
        }
        __syncthreads();
        for (int idx = tid; idx < ROWS * TILE / 8; idx += 64 * kWaves) {
            const int r = idx / (TILE / 8), cg = idx % (TILE / 8), m = m0 + half * ROWS + r, n = n0 + cg * 8;
            if (m >= M || n >= N) continue;
            float* dst = static_cast<float*>(pr.C) + (long long)m * N + n;
            float val[8] = {};
            const float* src = reinterpret_cast<const float*>(&lds[0][0][0]) + place(r, cg * 8);
            for (int w = 0; w < n_parts; w++) {
                const float4 lo = *reinterpret_cast<const float4*>(src + w * (kRing * STAGE / 2)), hi = *reinterpret_cast<const float4*>(src + w * (kRing * STAGE / 2) + 4);
                val[0] += lo.x; val[1] += lo.y; val[2] += lo.z; val[3] += lo.w;
                val[4] += hi.x; val[5] += hi.y; val[6] += hi.z; val[7] += hi.w;
            }
            float4 lo = make_float4(val[0], val[1], val[2], val[3]), hi = make_float4(val[4], val[5], val[6], val[7]);
            if (pr.accumulate) {
                const float4 o0 = reinterpret_cast<const float4*>(dst)[0], o1 = reinterpret_cast<const float4*>(dst)[1];
                lo.x += o0.x; lo.y += o0.y; lo.z += o0.z; lo.w += o0.w;
                hi.x += o1.x; hi.y += o1.y; hi.z += o1.z; hi.w += o1.w;
            }
            reinterpret_cast<float4*>(dst)[0] = lo;
            reinterpret_cast<float4*>(dst)[1] = hi;
        }
    }
}

}  // namespace

void eisen_gemm_launch_dw(eisen_ctx* ctx, const DwArgs& g, int tile) {
    if (tile == 128) gemm_dw_kernel<128><<<(unsigned)g.tiles, 64 * kWaves, 0, ctx->stream>>>(g);
    else gemm_dw_kernel<64><<<(unsigned)g.tiles, 64 * kWaves, 0, ctx->stream>>>(g);
}

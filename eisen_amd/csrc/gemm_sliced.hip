// bf16 GEMM for any shape, 64 x 64 or 32 x 32 tiles whose contraction is dealt to the waves of the workgroup (f32 accumulate).
//
// The kernels of gemm.hip and gemm_wide.hip want whole tiles of 128 or 256 and enough of them to fill 256 CUs.  This one takes the
// rest: odd batch and sequence lengths, head and vocabulary sizes that are no multiple of anything, and products with few
// output tiles, whose time is latency (a wave of a shared tile waits for memory, then for a barrier, once per slab, with one
// workgroup on the CU).  Here a wave owns the whole tile for every W-th 64-deep slice of the contraction and a private
// 16 KB (8 KB) of LDS filled by direct-to-LDS loads: no barrier in the loop, W independent chains per CU that cover each other's waits.  A
// slice is read into registers as a whole, the loads of the wave's next one go out, and its 16 (4) MFMAs run under them.  The W partial
// tiles meet in LDS once, where a thread ends up with eight consecutive columns of a row, so every epilogue works on 16-byte packets.
//
// What bounds it: a CU fetches 256 bytes per contraction index for its tile, from an L2 that gives it about 40 bytes per clock; the
// matrix cores would need 4 clocks for what that takes 6.  Long contractions of one tile per CU run at 0.6 PFLOP/s for that
// reason, short ones at their latency (launch, first slice, meeting).  us with operands from memory, slices 32 deep in a two-stage
// ring / now: 1024 x 1024 x 1024 NT 8.4 / 7.3, NN 9.0 / 7.9, x 4096 NT in two segments 22.5 / 18.2; 2048 x 768 x 4096 38.4 / 29.0;
// 8192 x 256 x 256 7.6 / 6.5; 512 x 768 x 768 7.3 / 6.3; 201 x 256 x 1024 7.7 / 6.6; weight gradients 768 x 768 x 2048 12.6 / 12.0.  Tiles of 32
// where there are few of 64: the same latency over four times the workgroups with a quarter of the work each (201 x 256 x 1024 6.6 -> 5.2; figures at the rule in
// gemm.hip).
//
// Edges.  Rows (m, n) past the end re-read the last row or chunk: they only reach outputs that are not stored.  Contraction
// indices past the end of a segment re-read the last one, and both fragments are zeroed there.  Operand rows must start on
// 16-byte boundaries and be readable up to the next multiple of 8 elements (the caller packs operands that are not).
#include "gemm_common.cuh"

namespace {

constexpr int SK = 64;  // depth of a slice

// One operand of a slice, ST x 64 elements, into the LDS, in loads of 1 KB: rows of 128 bytes, whole cache lines, except for tiles of 32 of an operand
// that is stored along its rows.  (Slices 32 deep read half a line at a time of an operand stored along the contraction; the other half
// belonged to the next wave, and the L1 had dropped the line by then more often than not: 1.5 times the L2 reads, which is what bounds this
// kernel for long contractions.)
// The rows are operand rows or contraction indices, whichever way the operand is stored; row_last, chunk_last: the last ones that exist.
template <int ST, bool KC>
__device__ __forceinline__ void load_slice(const bf16_t* base, int ld, unsigned tile, int row_last, int chunk_last, int lane) {
    constexpr int CPR = KC ? 8 : ST / 8, RPL = 64 / CPR, LOADS = ST / 8;  // 16-byte chunks per row, rows per load, loads
    const int row = lane / CPR;  // of load 0
    if (row_last >= RPL * LOADS - 1 && chunk_last >= CPR - 1) {
        unsigned off[2];  // (the permutation of the chunks repeats after 16 rows)
#pragma unroll
        for (int odd = 0; odd < 2; odd++) off[odd] = (unsigned)(row * ld + ((lane % CPR) ^ lds_swz<CPR * 16>(row + 8 * odd)) * 8) * 2u;
        static_for<LOADS>([&](auto i_c) {
            constexpr int i = decltype(i_c)::value;
            load_to_lds_16_at<i * 1024>(base + (long long)i * RPL * ld, off[RPL == 8 ? i & 1 : 0], tile);
        });
    } else {
        static_for<LOADS>([&](auto i_c) {
            constexpr int i = decltype(i_c)::value;
            const int r = row + RPL * i, chunk = (lane % CPR) ^ lds_swz<CPR * 16>(r);
            load_to_lds_16_at<i * 1024>(base, (unsigned)(min(r, row_last) * ld + min(chunk, chunk_last) * 8) * 2u, tile);
        });
    }
}

// The same for 32 columns each of two operands [K][N] side by side: the first four chunks of a row are the first one's.
__device__ __forceinline__ void load_slice_of_two(const bf16_t* first, const bf16_t* second, int ld, unsigned tile, int row_last, int chunk_last, int lane) {
    static_for<8>([&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        const int row = (lane >> 3) + 8 * i, chunk = (lane & 7) ^ lds_swz<128>(row);
        load_to_lds_16_at<i * 1024>((chunk < 4 ? first : second) + (long long)(min(row, row_last) * ld + min(chunk & 3, chunk_last) * 8), tile);
    });
}

// integer divisions leave values that are the same in every lane in vector registers
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

enum class Kind { kPlain, kSegments, kGroup, kSwiglu };

template <int W, int ST, bool A_KC, bool B_KC, typename TC, Kind KIND>
__global__ __launch_bounds__(64 * W) void gemm_sliced_kernel(GemmArgs g) {
    using TA = DirectOperandTile<ST, A_KC, SK, 1>;
    using TB = DirectOperandTile<ST, B_KC, SK, 1>;
    constexpr int STAGE = TA::ELEMS + TB::ELEMS, STEPS = SK / 16, TM = ST / 32;
    static_assert(KIND != Kind::kSwiglu || ST == 64, "32 columns of each product");
    static_assert(STAGE * sizeof(bf16_t) >= ST * ST * sizeof(float), "a wave's partial tile takes the place of its slice");
    __shared__ __attribute__((aligned(1024))) bf16_t lds[W][STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blocks of 4 x 8 tiles, which share 12 operand panels, on one XCD
    const int split = g.split > 1 ? g.split : 1;
    int nt, mt = 0, zz, member = 0;
    if constexpr (KIND == Kind::kGroup) {  // which product this tile belongs to (uniform); static indices keep the tables in scalar registers
        const int tiles = g.grp_tile_end[kMaxGroup - 1];
        const int lin = xcd_contiguous_id(blockIdx.x, tiles * split);
        zz = uniform(lin / tiles);
        const int t = lin - zz * tiles;
        int first = 0;
        long long partial_off = g.grp_partial_off[0];
        g.A = g.grp_A[0]; g.B = g.grp_B[0]; g.C = g.grp_C[0]; g.N = g.grp_N[0];
#pragma unroll
        for (int q = 1; q < kMaxGroup; q++)
            if (t >= g.grp_tile_end[q - 1]) {
                member = q;
                first = g.grp_tile_end[q - 1];
                partial_off = g.grp_partial_off[q];
                g.A = g.grp_A[q]; g.B = g.grp_B[q]; g.C = g.grp_C[q]; g.N = g.grp_N[q];
            }
        if (split > 1) g.partial += partial_off;
        const int n_tiles = (g.N + ST - 1) / ST;
        mt = (t - first) / n_tiles;
        nt = (t - first) % n_tiles;
        g.ldc = g.N;
        if (!B_KC) g.ldb = g.N;
    } else {
        constexpr int COLS = KIND == Kind::kSwiglu ? ST / 2 : ST;  // columns of each product
        const int gx = (g.N + COLS - 1) / COLS, gy = (g.M + ST - 1) / ST;
        const int lin = xcd_contiguous_id(blockIdx.x, g.blocks);
        zz = uniform(lin / (gx * gy));
        block_tile<4, 8>(lin - zz * (gx * gy), gy, gx, mt, nt);
    }
    const int m0 = uniform(mt * ST), n0 = uniform(nt * (KIND == Kind::kSwiglu ? ST / 2 : ST));
    const int bz = uniform(zz / split), part = uniform(zz % split);
    if constexpr (KIND != Kind::kGroup) member = bz;
    const bf16_t* A = static_cast<const bf16_t*>(g.A) + (long long)bz * g.sA;
    const bf16_t* B = static_cast<const bf16_t*>(g.B) + (long long)bz * g.sB;

    // Slices of the contraction: segment by segment, each with a last slice of its own.  This workgroup's are [s_lo, s_hi).
    constexpr bool SEG = KIND == Kind::kSegments;
    const int len0 = SEG ? g.seg_end[0] : g.K;
    const int sl0 = (len0 + SK - 1) / SK;
    const int len1 = !SEG ? 0 : g.nseg > 2 ? g.seg_end[1] - g.seg_end[0] : g.K - g.seg_end[0], sl1 = (len1 + SK - 1) / SK;
    const int len2 = SEG && g.nseg > 2 ? g.K - g.seg_end[1] : 0, sl2 = (len2 + SK - 1) / SK;
    const bf16_t *A1 = nullptr, *A2 = nullptr, *B1 = nullptr, *B2 = nullptr;
    int lda1 = 0, lda2 = 0, ldb1 = 0, ldb2 = 0;
    const int lda0 = g.lda, ldb0 = g.ldb;
    if constexpr (SEG) {
        A1 = static_cast<const bf16_t*>(g.A_seg[0]); A2 = static_cast<const bf16_t*>(g.A_seg[1]);
        B1 = static_cast<const bf16_t*>(g.B_seg[0]); B2 = static_cast<const bf16_t*>(g.B_seg[1]);
        lda1 = g.lda_seg[0]; lda2 = g.lda_seg[1];
        ldb1 = g.ldb_seg[0]; ldb2 = g.ldb_seg[1];
    }
    const int s_lo = part * (g.k_part / SK), s_hi = split > 1 ? min(sl0, s_lo + g.k_part / SK) : sl0 + sl1 + sl2;
    const int n_mine = s_hi - s_lo > wave ? (s_hi - s_lo - wave + W - 1) / W : 0;
    const int n_parts = min(W, s_hi - s_lo);  // waves with something to add

    bf16_t* As = lds[wave];
    bf16_t* Bs = As + TA::ELEMS;
    const int m_last = g.M - 1 - m0, n_last = g.N - 1 - n0;  // last row of the tile that exists
    const unsigned lds_a = uniform((int)(size_t)(lds_void_ptr)As), lds_b = lds_a + TA::ELEMS * 2;  // their LDS addresses
    // the loads of this wave's i-th slice; returns how many of its contraction indices exist
    auto issue = [&](int i) __attribute__((always_inline)) -> int {
        int s = s_lo + wave + i * W, lda = lda0, ldb = ldb0, len = len0;
        const bf16_t* Ap = A;
        const bf16_t* Bp = B;
        if (SEG && s >= sl0) {
            s -= sl0;
            Ap = A1; Bp = B1; lda = lda1; ldb = ldb1; len = len1;
            if (s >= sl1) {
                s -= sl1;
                Ap = A2; Bp = B2; lda = lda2; ldb = ldb2; len = len2;
            }
        }
        const int k0 = s * SK, left = len - k0;
        load_slice<ST, A_KC>(A_KC ? Ap + (long long)m0 * lda + k0 : Ap + (long long)k0 * lda + m0, lda, lds_a, A_KC ? m_last : left - 1, (A_KC ? left - 1 : m_last) / 8, lane);
        if constexpr (KIND == Kind::kSwiglu)
            load_slice_of_two(Bp + (long long)k0 * ldb + n0, static_cast<const bf16_t*>(g.B_seg[0]) + (long long)k0 * ldb + n0, ldb, lds_b, left - 1, n_last / 8, lane);
        else
            load_slice<ST, B_KC>(B_KC ? Bp + (long long)n0 * ldb + k0 : Bp + (long long)k0 * ldb + n0, ldb, lds_b, B_KC ? n_last : left - 1, (B_KC ? left - 1 : n_last) / 8, lane);
        return min(left, SK);
    };

    int left = 0;
    if (n_mine > 0) left = issue(0);

    // What the epilogue reads (the old C or the residual; gate and up) is requested behind the first slice (in front of it, the branches
    // around these loads would make every wave wait for them before it asks for an operand).
    constexpr int GROUPS = ST * ST / 8, PASSES = (GROUPS + 64 * W - 1) / (64 * W);  // groups of eight columns: of the tile, per thread
    TC* C = static_cast<TC*>(g.C) + (long long)bz * g.sC;
    const TC* Rsrc = g.R ? static_cast<const TC*>(g.R) + (long long)bz * g.sC : C;
    float* P = gemm_partial<TC>(g, bz, split, part);
    const bool add_old = KIND != Kind::kSwiglu && (g.accumulate || g.R != nullptr) && !P && !g.gate;
    typename Eight<TC>::V first[PASSES] = {}, second[PASSES] = {};
    static_for<PASSES>([&](auto ps_c) {
        constexpr int ps = decltype(ps_c)::value;
        const int idx = ps * 64 * W + tid, m = m0 + idx / (ST / 8), n = n0 + (idx % (ST / 8)) * 8;
        const bool whole = KIND != Kind::kSwiglu && idx < GROUPS && m < g.M && n + 8 <= g.N;
        const long long at = (long long)m * g.ldc + n;
        if (whole && add_old) first[ps] = load_eight(Rsrc + at);
        if (whole && g.gate) {
            first[ps] = load_eight(static_cast<const TC*>(g.gate) + (long long)bz * g.sC + at);
            second[ps] = load_eight(static_cast<const TC*>(g.up) + (long long)bz * g.sC + at);
        }
    });

    f32x16 acc[TM][TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    for (int i = 0; i < n_mine; i++) {
        wait_loads_but<0>();
        bf16x8 a[STEPS][TM], b[STEPS][TM];
#pragma unroll
        for (int st = 0; st < STEPS; st++)
#pragma unroll
            for (int h = 0; h < TM; h++) {
                a[st][h] = TA::fragment(As, h * 32, st * 16, lane);
                b[st][h] = TB::fragment(Bs, h * 32, st * 16, lane);
            }
        const int now = left;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slice is in registers: the next one may overwrite it
        if (i + 1 < n_mine) left = issue(i + 1);
        if (now < SK) {
#pragma unroll
            for (int st = 0; st < STEPS; st++)
#pragma unroll
                for (int h = 0; h < TM; h++) {
                    const int k = st * 16 + 8 * (lane >> 5);
                    a[st][h] = zero_from(a[st][h], k, now);
                    b[st][h] = zero_from(b[st][h], k, now);
                }
        }
#pragma unroll
        for (int st = 0; st < STEPS; st++)
#pragma unroll
            for (int p = 0; p < TM; p++)
#pragma unroll
                for (int q = 0; q < TM; q++) acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st][p], b[st][q], acc[p][q], 0, 0, 0);
    }

    // The waves' tiles, each in the place of its (now idle) slice, rows 4 apart (the two halves of a wave) in different halves of the banks.
    auto place = [](int r, int n) { return ST == 64 ? r * 64 + (n ^ ((r >> 2 & 1) * 32)) : (r ^ (r >> 2 & 1)) * 32 + n; };
    float* mine = reinterpret_cast<float*>(As);
    if (n_mine > 0) {
        const int c = lane & 31, gh = lane >> 5;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) mine[place(i * 32 + 8 * (v / 4) + 4 * gh + (v % 4), j * 32 + c)] = acc[i][j][v];
    }
    __syncthreads();
    auto sum_of_waves = [&](int r, int cg, float (&val)[8]) __attribute__((always_inline)) {
        const float* src = reinterpret_cast<const float*>(lds[0]) + place(r, cg * 8);
#pragma unroll
        for (int e = 0; e < 8; e++) val[e] = 0.f;
        for (int w = 0; w < n_parts; w++) {  // in wave order
            const float4 lo = *reinterpret_cast<const float4*>(src + w * (STAGE / 2)), hi = *reinterpret_cast<const float4*>(src + w * (STAGE / 2) + 4);
            val[0] += lo.x; val[1] += lo.y; val[2] += lo.z; val[3] += lo.w;
            val[4] += hi.x; val[5] += hi.y; val[6] += hi.z; val[7] += hi.w;
        }
    };
    if constexpr (KIND == Kind::kSwiglu) {
        // G = X Wg and U = X Wu leave rounded, and H = silu(G) * U is formed from what was rounded, as a separate kernel would
        const int idx = tid, r = idx / 4, cg = idx % 4, m = m0 + r, n = n0 + cg * 8;
        if (idx >= ST * 4 || m >= g.M || n >= g.N) return;
        float gv[8], uv[8];
        sum_of_waves(r, cg, gv);
        sum_of_waves(r, cg + 4, uv);
        bf16x8 og, ou, oh;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            og[e] = (bf16_t)gv[e];
            ou[e] = (bf16_t)uv[e];
            const float x = (float)og[e];
            oh[e] = (bf16_t)(x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)) * (float)ou[e]);  // 1-ulp reciprocal: the result is rounded to bf16
        }
        const long long at = (long long)m * g.N + n;  // (N is a multiple of 8 and the results start on 16-byte boundaries)
        *reinterpret_cast<bf16x8*>(static_cast<bf16_t*>(g.C) + at) = og;
        *reinterpret_cast<bf16x8*>(static_cast<bf16_t*>(g.C2) + at) = ou;
        *reinterpret_cast<bf16x8*>(static_cast<bf16_t*>(g.grp_C[0]) + at) = oh;
    } else {
        static_for<PASSES>([&](auto ps_c) {
            constexpr int ps = decltype(ps_c)::value;
            const int idx = ps * 64 * W + tid, r = idx / (ST / 8), cg = idx % (ST / 8);
            const int m = m0 + r, n = n0 + cg * 8;
            if (idx >= GROUPS || m >= g.M || n >= g.N) return;
            float val[8];
            sum_of_waves(r, cg, val);
            gemm_store_eight<TC>(g, val, m, n, member, C, Rsrc, add_old, P, first[ps], second[ps]);
        });
    }
}

template <int W, typename TC, Kind KIND>
void launch_sliced(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc) {
    const unsigned grid = (unsigned)g.blocks;
    if (a_kc && b_kc) gemm_sliced_kernel<W, 64, true, true, TC, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g);
    else if (a_kc) gemm_sliced_kernel<W, 64, true, false, TC, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g);
    else if (b_kc) gemm_sliced_kernel<W, 64, false, true, TC, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g);
    else gemm_sliced_kernel<W, 64, false, false, TC, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g);
}
// 32 x 32 tiles: products with A stored along the contraction, and weight gradients
template <int W, typename TC, Kind KIND>
void launch_sliced_32(eisen_ctx* ctx, const GemmArgs& g, bool b_kc) {
    if (b_kc) gemm_sliced_kernel<W, 32, true, true, TC, KIND><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
    else gemm_sliced_kernel<W, 32, true, false, TC, KIND><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
}
template <int W>
void launch_sliced_32_w(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc, int dtype_c) {
    if (!a_kc && g.ngroup > 0) gemm_sliced_kernel<W, 32, false, false, float, Kind::kGroup><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
    else if (!a_kc) gemm_sliced_kernel<W, 32, false, false, float, Kind::kPlain><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
    else if (g.ngroup > 0) gemm_sliced_kernel<W, 32, true, false, bf16_t, Kind::kGroup><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
    else if (g.nseg > 1 && dtype_c == EISEN_BF16) launch_sliced_32<W, bf16_t, Kind::kSegments>(ctx, g, b_kc);
    else if (g.nseg > 1) launch_sliced_32<W, float, Kind::kSegments>(ctx, g, b_kc);
    else if (dtype_c == EISEN_BF16) launch_sliced_32<W, bf16_t, Kind::kPlain>(ctx, g, b_kc);
    else launch_sliced_32<W, float, Kind::kPlain>(ctx, g, b_kc);
}
template <int W>
void launch_sliced_w(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc, int dtype_c) {
    if (g.ngroup > 0 && dtype_c == EISEN_BF16) gemm_sliced_kernel<W, 64, true, false, bf16_t, Kind::kGroup><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
    else if (g.ngroup > 0) gemm_sliced_kernel<W, 64, false, false, float, Kind::kGroup><<<(unsigned)g.blocks, 64 * W, 0, ctx->stream>>>(g);
    else if (g.nseg > 1 && dtype_c == EISEN_BF16) launch_sliced<W, bf16_t, Kind::kSegments>(ctx, g, a_kc, b_kc);
    else if (g.nseg > 1) launch_sliced<W, float, Kind::kSegments>(ctx, g, a_kc, b_kc);
    else if (dtype_c == EISEN_BF16) launch_sliced<W, bf16_t, Kind::kPlain>(ctx, g, a_kc, b_kc);
    else launch_sliced<W, float, Kind::kPlain>(ctx, g, a_kc, b_kc);
}

}  // namespace

// Grouped launches (g.ngroup > 0) are weight gradients (both operands stored along their rows, f32 results) or forward products (A
// stored along the contraction, B along its rows, bf16 results).
void eisen_gemm_launch_sliced(eisen_ctx* ctx, GemmArgs g, int waves, int tile, bool a_kc, bool b_kc, int batch, int dtype_c) {
    const int split = g.split > 1 ? g.split : 1;
    if (g.ngroup > 0) {
        for (int p = g.ngroup; p < kMaxGroup; p++) g.grp_tile_end[p] = g.grp_tile_end[g.ngroup - 1];  // no tile belongs to the missing ones
        g.blocks = g.grp_tile_end[kMaxGroup - 1] * split;
    } else {
        g.blocks = (int)eisen_ceil_div(g.M, tile) * (int)eisen_ceil_div(g.N, tile) * batch * split;
    }
    if (tile == 64 && waves == 8) launch_sliced_w<8>(ctx, g, a_kc, b_kc, dtype_c);
    else if (tile == 64) launch_sliced_w<4>(ctx, g, a_kc, b_kc, dtype_c);
    else if (waves == 8) launch_sliced_32_w<8>(ctx, g, a_kc, b_kc, dtype_c);
    else launch_sliced_32_w<4>(ctx, g, a_kc, b_kc, dtype_c);
}

// G = X Wg, U = X Wu, H = silu(G) * U: A = X [M][K], B = Wg and B_seg[0] = Wu [K][N], C = G, C2 = U, grp_C[0] = H.
void eisen_gemm_launch_sliced_swiglu(eisen_ctx* ctx, GemmArgs g, int waves) {
    g.blocks = (int)eisen_ceil_div(g.M, 64) * (int)eisen_ceil_div(g.N, 32);
    if (waves == 8) gemm_sliced_kernel<8, 64, true, false, bf16_t, Kind::kSwiglu><<<(unsigned)g.blocks, 512, 0, ctx->stream>>>(g);
    else gemm_sliced_kernel<4, 64, true, false, bf16_t, Kind::kSwiglu><<<(unsigned)g.blocks, 256, 0, ctx->stream>>>(g);
}

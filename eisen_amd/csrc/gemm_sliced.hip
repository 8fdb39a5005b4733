// bf16 GEMM for any shape, 64 x 64 tiles whose contraction is dealt to the waves of the workgroup (f32 accumulate).
//
// The kernels of gemm.hip and gemm_wide.hip want whole tiles of 128 or 256 and enough of them to fill 256 CUs.  This one takes the
// rest: odd batch and sequence lengths, head and vocabulary sizes that are no multiple of anything, and products with few
// output tiles, whose time is latency (a wave of a shared tile waits for memory, then for a barrier, once per slab, with one
// workgroup on the CU).  Here a wave owns the whole 64 x 64 tile for every W-th 32-deep slice of the contraction and a private
// two-stage LDS ring filled by direct-to-LDS loads: no barrier in the loop, W independent chains per CU that cover each other's
// waits, and even K = 256 keeps all of them busy.  The W partial tiles meet in LDS once, where a thread ends up with eight
// consecutive columns of a row, so every epilogue works on 16-byte packets.  The price is LDS traffic (every operand byte is
// written and read once per 64 x 64 tile and slice), which caps it near half of the matrix rate.
//
// Edges.  Rows (m, n) past the end re-read the last row or chunk: they only reach outputs that are not stored.  Contraction
// indices past the end of a segment re-read the last one, and both fragments are zeroed there.  Operand rows must start on
// 16-byte boundaries and be readable up to the next multiple of 8 elements (the caller packs operands that are not).
#include "gemm_common.cuh"

namespace {

constexpr int ST = 64, SK = 32;  // tile rows and columns, depth of a slice

template <int W, bool A_KC, bool B_KC, typename TC>
__global__ __launch_bounds__(64 * W) void gemm_sliced_kernel(GemmArgs g) {
    using TA = DirectOperandTile<ST, A_KC, SK, 1>;
    using TB = DirectOperandTile<ST, B_KC, SK, 1>;
    constexpr int NLOADS = TA::LOADS + TB::LOADS, STAGE = TA::ELEMS + TB::ELEMS;
    static_assert(2 * STAGE * sizeof(bf16_t) == ST * ST * sizeof(float), "a wave's partial tile takes the place of its ring");
    __shared__ __attribute__((aligned(1024))) bf16_t lds[W][2 * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blocks of 4 x 8 tiles, which share 12 operand panels, on one XCD
    const int gx = gridDim.x, gy = gridDim.y;
    const int lin = xcd_contiguous_id(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), gx * gy * gridDim.z);
    const int zz = lin / (gx * gy);
    int nt = lin % (gx * gy), mt = 0;
    if (g.ngroup == 0) block_tile<4, 8>(nt, gy, gx, mt, nt);
    if (g.ngroup > 0) {  // which product this tile belongs to (uniform); static indices keep the tables in scalar registers
        const int t = nt;
        int first = 0;
        long long partial_off = g.grp_partial_off[0];
        g.A = g.grp_A[0]; g.B = g.grp_B[0]; g.C = g.grp_C[0]; g.N = g.grp_N[0];
#pragma unroll
        for (int q = 1; q < kMaxGroup; q++)
            if (q < g.ngroup && t >= g.grp_tile_end[q - 1]) {
                first = g.grp_tile_end[q - 1];
                partial_off = g.grp_partial_off[q];
                g.A = g.grp_A[q]; g.B = g.grp_B[q]; g.C = g.grp_C[q]; g.N = g.grp_N[q];
            }
        if (g.split > 1) g.partial += partial_off;
        const int n_tiles = (g.N + ST - 1) / ST;
        mt = (t - first) / n_tiles;
        nt = (t - first) % n_tiles;
        g.ldc = g.N;
        if (!B_KC) g.ldb = g.N;
    }
    const int m0 = mt * ST, n0 = nt * ST;
    const int split = g.split > 1 ? g.split : 1;
    const int bz = zz / split, part = zz % split;
    const bf16_t* A = static_cast<const bf16_t*>(g.A) + (long long)bz * g.sA;
    const bf16_t* B = static_cast<const bf16_t*>(g.B) + (long long)bz * g.sB;

    // Slices of the contraction: segment by segment, each with a last slice of its own.  This workgroup's are [s_lo, s_hi).
    const int len0 = g.nseg > 1 ? g.seg_end[0] : g.K;
    const int sl0 = (len0 + SK - 1) / SK;
    const int len1 = g.nseg > 2 ? g.seg_end[1] - g.seg_end[0] : g.nseg > 1 ? g.K - g.seg_end[0] : 0, sl1 = (len1 + SK - 1) / SK;
    const int len2 = g.nseg > 2 ? g.K - g.seg_end[1] : 0, sl2 = (len2 + SK - 1) / SK;
    const int s_lo = part * (g.k_part / SK), s_hi = split > 1 ? min(sl0, s_lo + g.k_part / SK) : sl0 + sl1 + sl2;
    const int n_mine = s_hi - s_lo > wave ? (s_hi - s_lo - wave + W - 1) / W : 0;
    const int n_parts = min(W, s_hi - s_lo);  // waves with something to add

    // What the epilogue reads (the old C or the residual; gate and up) is requested first.
    constexpr int PASSES = ST * ST / 8 / (64 * W);               // groups of eight columns per thread
    TC* C = static_cast<TC*>(g.C) + (long long)bz * g.sC;
    const TC* Rsrc = g.R ? static_cast<const TC*>(g.R) + (long long)bz * g.sC : C;
    float* P = gemm_partial<TC>(g, bz, split, part);
    const bool add_old = (g.accumulate || g.R != nullptr) && !P && !g.gate;
    using Eight = LooseEight<TC>;
    Eight first[PASSES], second[PASSES];
#pragma unroll
    for (int ps = 0; ps < PASSES; ps++) {
        const int idx = ps * 64 * W + tid, m = m0 + idx / 8, n = n0 + (idx % 8) * 8;
        const bool whole = m < g.M && n + 8 <= g.N;
        const long long at = (long long)m * g.ldc + n;
        if (whole && add_old) first[ps] = *reinterpret_cast<const Eight*>(Rsrc + at);
        if (whole && g.gate) {
            first[ps] = *reinterpret_cast<const Eight*>(static_cast<const TC*>(g.gate) + (long long)bz * g.sC + at);
            second[ps] = *reinterpret_cast<const Eight*>(static_cast<const TC*>(g.up) + (long long)bz * g.sC + at);
        }
    }

    int a_row[TA::LOADS], a_chunk[TA::LOADS], b_row[TB::LOADS], b_chunk[TB::LOADS];
    unsigned a_off[TA::LOADS], b_off[TB::LOADS];
    const int m_last = g.M - 1 - m0, n_last = g.N - 1 - n0;  // last row of the tile that exists
#pragma unroll
    for (int i = 0; i < TA::LOADS; i++) {
        TA::lane_chunk(i, 0, lane, a_row[i], a_chunk[i]);
        if (A_KC) a_row[i] = min(a_row[i], m_last);
        else a_chunk[i] = min(a_chunk[i], m_last / 8);
    }
#pragma unroll
    for (int i = 0; i < TB::LOADS; i++) {
        TB::lane_chunk(i, 0, lane, b_row[i], b_chunk[i]);
        if (B_KC) b_row[i] = min(b_row[i], n_last);
        else b_chunk[i] = min(b_chunk[i], n_last / 8);
    }
    int off_lda = -1, off_ldb = -1;
    auto set_offsets = [&](int lda, int ldb) {
        if (lda != off_lda) {
#pragma unroll
            for (int i = 0; i < TA::LOADS; i++) a_off[i] = (unsigned)(a_row[i] * lda + a_chunk[i] * 8) * 2u;
            off_lda = lda;
        }
        if (ldb != off_ldb) {
#pragma unroll
            for (int i = 0; i < TB::LOADS; i++) b_off[i] = (unsigned)(b_row[i] * ldb + b_chunk[i] * 8) * 2u;
            off_ldb = ldb;
        }
    };
    bf16_t* ring = lds[wave];
    // the loads of this wave's i-th slice into ring stage i % 2; returns how many of its contraction indices exist
    auto issue = [&](int i) -> int {
        int s = s_lo + wave + i * W, lda = g.lda, ldb = g.ldb, len = len0;
        const bf16_t* Ap = A;
        const bf16_t* Bp = B;
        if (g.nseg > 1) {
            const bool s1 = s >= sl0, s2 = g.nseg > 2 && s >= sl0 + sl1;
            Ap = s2 ? static_cast<const bf16_t*>(g.A_seg[1]) : s1 ? static_cast<const bf16_t*>(g.A_seg[0]) : A;
            Bp = s2 ? static_cast<const bf16_t*>(g.B_seg[1]) : s1 ? static_cast<const bf16_t*>(g.B_seg[0]) : B;
            lda = s2 ? g.lda_seg[1] : s1 ? g.lda_seg[0] : lda;
            ldb = s2 ? g.ldb_seg[1] : s1 ? g.ldb_seg[0] : ldb;
            len = s2 ? len2 : s1 ? len1 : len0;
            s -= s2 ? sl0 + sl1 : s1 ? sl0 : 0;
        }
        const int k0 = s * SK, left = len - k0;
        const bf16_t* a0 = A_KC ? Ap + (long long)m0 * lda + k0 : Ap + (long long)k0 * lda + m0;
        const bf16_t* b0 = B_KC ? Bp + (long long)n0 * ldb + k0 : Bp + (long long)k0 * ldb + n0;
        bf16_t* As = ring + (i & 1) * STAGE;
        bf16_t* Bs = As + TA::ELEMS;
        set_offsets(lda, ldb);
        if (left >= SK) {
#pragma unroll
            for (int h = 0; h < TA::LOADS; h++) load_to_lds_16(a0, a_off[h], As + TA::lds_block(h, 0));
#pragma unroll
            for (int h = 0; h < TB::LOADS; h++) load_to_lds_16(b0, b_off[h], Bs + TB::lds_block(h, 0));
            return SK;
        }
        const int last = left - 1;
#pragma unroll
        for (int h = 0; h < TA::LOADS; h++) {
            const int row = A_KC ? a_row[h] : min(a_row[h], last), chunk = A_KC ? min(a_chunk[h], last / 8) : a_chunk[h];
            load_to_lds_16(a0, (unsigned)(row * lda + chunk * 8) * 2u, As + TA::lds_block(h, 0));
        }
#pragma unroll
        for (int h = 0; h < TB::LOADS; h++) {
            const int row = B_KC ? b_row[h] : min(b_row[h], last), chunk = B_KC ? min(b_chunk[h], last / 8) : b_chunk[h];
            load_to_lds_16(b0, (unsigned)(row * ldb + chunk * 8) * 2u, Bs + TB::lds_block(h, 0));
        }
        return left;
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    int left[2] = {0, 0};
    if (n_mine > 0) left[0] = issue(0);
    if (n_mine > 1) left[1] = issue(1);
    for (int i = 0; i < n_mine; i++) {
        if (i + 1 < n_mine) wait_loads_but<NLOADS>();
        else wait_loads_but<0>();
        const bf16_t* As = ring + (i & 1) * STAGE;
        const bf16_t* Bs = As + TA::ELEMS;
        bf16x8 a[2][2], b[2][2];
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                a[st][h] = TA::fragment(As, h * 32, st * 16, lane);
                b[st][h] = TB::fragment(Bs, h * 32, st * 16, lane);
            }
        const int now = left[0];
        left[0] = left[1];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read: the slice after next may overwrite it
        if (i + 2 < n_mine) left[1] = issue(i + 2);
        if (now < SK) {
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int k = st * 16 + 8 * (lane >> 5);
                    a[st][h] = zero_from(a[st][h], k, now);
                    b[st][h] = zero_from(b[st][h], k, now);
                }
        }
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int q = 0; q < 2; q++) acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st][p], b[st][q], acc[p][q], 0, 0, 0);
    }

    // The waves' tiles, each in the place of its (now idle) ring: row r, column n at r * 64 + ((n / 32) ^ (r / 4 % 2)) * 32 + n % 32,
    // so that the two halves of a wave (rows 4 apart) write to different banks.
    float* mine = reinterpret_cast<float*>(ring);
    if (n_mine > 0) {
        const int c = lane & 31, gh = lane >> 5;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) mine[(i * 32 + 8 * (v / 4) + 4 * gh + (v % 4)) * ST + (j ^ gh) * 32 + c] = acc[i][j][v];
    }
    __syncthreads();
#pragma unroll
    for (int ps = 0; ps < PASSES; ps++) {
        const int idx = ps * 64 * W + tid, r = idx / 8, cg = idx % 8;
        const int m = m0 + r, n = n0 + cg * 8;
        if (m >= g.M || n >= g.N) continue;
        const float* src = reinterpret_cast<const float*>(lds[0]) + r * ST + ((cg >> 2) ^ ((r >> 2) & 1)) * 32 + (cg & 3) * 8;
        float val[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int w = 0; w < n_parts; w++) {  // in wave order
            const float4 lo = *reinterpret_cast<const float4*>(src + w * ST * ST), hi = *reinterpret_cast<const float4*>(src + w * ST * ST + 4);
            val[0] += lo.x; val[1] += lo.y; val[2] += lo.z; val[3] += lo.w;
            val[4] += hi.x; val[5] += hi.y; val[6] += hi.z; val[7] += hi.w;
        }
        gemm_store_eight<TC>(g, val, m, n, bz, C, Rsrc, add_old, P, first[ps], second[ps]);
    }
}

template <int W, typename TC>
void launch_sliced(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc, dim3 grid) {
    if (a_kc && b_kc) gemm_sliced_kernel<W, true, true, TC><<<grid, 64 * W, 0, ctx->stream>>>(g);
    else if (a_kc) gemm_sliced_kernel<W, true, false, TC><<<grid, 64 * W, 0, ctx->stream>>>(g);
    else if (b_kc) gemm_sliced_kernel<W, false, true, TC><<<grid, 64 * W, 0, ctx->stream>>>(g);
    else gemm_sliced_kernel<W, false, false, TC><<<grid, 64 * W, 0, ctx->stream>>>(g);
}

}  // namespace

void eisen_gemm_launch_sliced(eisen_ctx* ctx, const GemmArgs& g, int waves, bool a_kc, bool b_kc, int batch, int dtype_c, unsigned group_tiles) {
    const dim3 grid(g.ngroup > 0 ? group_tiles : (unsigned)eisen_ceil_div(g.N, ST), g.ngroup > 0 ? 1u : (unsigned)eisen_ceil_div(g.M, ST),
                    (unsigned)(batch * (g.split > 1 ? g.split : 1)));
    if (waves == 8) {
        if (dtype_c == EISEN_BF16) launch_sliced<8, bf16_t>(ctx, g, a_kc, b_kc, grid);
        else launch_sliced<8, float>(ctx, g, a_kc, b_kc, grid);
    } else {
        if (dtype_c == EISEN_BF16) launch_sliced<4, bf16_t>(ctx, g, a_kc, b_kc, grid);
        else launch_sliced<4, float>(ctx, g, a_kc, b_kc, grid);
    }
}

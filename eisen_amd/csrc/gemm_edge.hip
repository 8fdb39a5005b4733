// bf16 GEMM for large products that are no whole tiles: 256 x 128 or 128 x 128 tiles of eight waves, slabs of 64, operands loaded
// straight into three LDS stages as in gemm_mfma_direct_kernel (gemm.hip), with bounds.
//
// A bound costs the main loop nothing.  Rows (m, n) past the end re-read the last row or chunk (they only reach outputs that are not
// stored): the byte offset a lane adds to a slab's origin is clamped once.  A slab that reaches past the end of its contraction or
// segment re-reads the last index; its offsets are formed anew when it is requested, and it runs a body of its own, which puts zeros
// in place of what does not exist in both operands' registers.  Operand rows must start on 16-byte boundaries and be readable up to the
// next multiple of 8 elements (the caller packs operands that are not); leading dimensions are below 2^22.
//
// What bounds it: rounds of workgroups (one per CU), and per slab the same as the kernel without bounds.  us, the register-staged kernel that ran these shapes /
// here: 4000 x 1000 x 1000 33.5 / 20.5, x 3000 NT 83 / 47, 7000 x 720 x 2000 66 / 47, 3840 x 3096 x 1024 58 / 48, 3840 x 1024 x (3096 + 3096) 176 / 93, weight
// gradients 1000 x 4000 x 4000 103 / 52, 8000 x 520 x 3000 84 / 54; 3000 x 8000 x 520 56 / 53.
#include "gemm_common.cuh"

namespace {

template <int BM, bool A_KC, bool B_KC, typename TC>
__global__ __launch_bounds__(512) void gemm_edge_kernel(GemmArgs g) {
    constexpr int BN = 128, BK = 64, WGM = 4, WGN = 2, WAVES = 8, STAGES = 3, KSTEPS = BK / 16;
    constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    using TA = DirectOperandTile<BM, A_KC, BK, WAVES>;
    using TB = DirectOperandTile<BN, B_KC, BK, WAVES>;
    constexpr int NLOADS = TA::LOADS + TB::LOADS;
    __shared__ __attribute__((aligned(1024))) bf16_t lds[STAGES][TA::ELEMS + TB::ELEMS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };  // integer divisions leave uniform values in vector registers
    const int split = g.split > 1 ? g.split : 1;
    const int gx = (g.N + BN - 1) / BN, gy = (g.M + BM - 1) / BM;
    const int lin = xcd_contiguous_id(blockIdx.x, g.blocks), zz = uniform(lin / (gx * gy));
    int mt, nt;
    block_tile<4, 8>(lin - zz * (gx * gy), gy, gx, mt, nt);  // blocks of 4 x 8 tiles, which share 12 operand panels, on one XCD
    const int m0 = uniform(mt * BM), n0 = uniform(nt * BN);
    const int bz = uniform(zz / split), part = uniform(zz % split);
    const int k_lo = part * g.k_part;
    const bf16_t* A0 = static_cast<const bf16_t*>(g.A) + (long long)bz * g.sA + (A_KC ? (long long)k_lo : (long long)k_lo * g.lda);
    const bf16_t* B0 = static_cast<const bf16_t*>(g.B) + (long long)bz * g.sB + (B_KC ? (long long)k_lo : (long long)k_lo * g.ldb);

    // slabs of the contraction: segment by segment, each with a last slab of its own
    const int len0 = split > 1 ? min(g.K, k_lo + g.k_part) - k_lo : g.nseg > 1 ? g.seg_end[0] : g.K;
    const int len1 = g.nseg > 2 ? g.seg_end[1] - g.seg_end[0] : g.nseg > 1 ? g.K - g.seg_end[0] : 0, len2 = g.nseg > 2 ? g.K - g.seg_end[1] : 0;
    const int sl0 = (len0 + BK - 1) / BK, sl1 = (len1 + BK - 1) / BK, nk = sl0 + sl1 + (len2 + BK - 1) / BK;
    const bf16_t *A1 = static_cast<const bf16_t*>(g.A_seg[0]), *A2 = static_cast<const bf16_t*>(g.A_seg[1]);
    const bf16_t *B1 = static_cast<const bf16_t*>(g.B_seg[0]), *B2 = static_cast<const bf16_t*>(g.B_seg[1]);
    const int lda0 = g.lda, ldb0 = g.ldb, lda1 = g.lda_seg[0], lda2 = g.lda_seg[1], ldb1 = g.ldb_seg[0], ldb2 = g.ldb_seg[1];

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    // this lane's chunk of each of its wave's loads, as a byte offset from the slab's origin: for the leading dimensions and the
    // number of contraction indices in force
    const int m_last = min(g.M - m0, BM) - 1, n_last = min(g.N - n0, BN) - 1;
    unsigned a_off[TA::LOADS], b_off[TB::LOADS];
    int off_lda = -1, off_ldb = -1, off_left = -1;
    auto set_offsets = [&](int lda, int ldb, int left) __attribute__((always_inline)) {
        if (lda == off_lda && ldb == off_ldb && left == off_left) return;
        off_lda = lda;
        off_ldb = ldb;
        off_left = left;
        const int k_last = left - 1;
#pragma unroll
        for (int i = 0; i < TA::LOADS; i++) {
            int row, chunk;
            TA::lane_chunk(i, wave, lane, row, chunk);
            a_off[i] = (unsigned)(min(row, A_KC ? m_last : k_last) * lda + min(chunk, (A_KC ? k_last : m_last) / 8) * 8) * 2u;
        }
#pragma unroll
        for (int i = 0; i < TB::LOADS; i++) {
            int row, chunk;
            TB::lane_chunk(i, wave, lane, row, chunk);
            b_off[i] = (unsigned)(min(row, B_KC ? n_last : k_last) * ldb + min(chunk, (B_KC ? k_last : n_last) / 8) * 8) * 2u;
        }
    };
    struct SlabSource {
        const bf16_t *a0, *b0;
        unsigned lds_a, lds_b;
    };
    // how many contraction indices of a slab exist
    auto left_of = [&](int s) __attribute__((always_inline)) { return min(BK, s < sl0 ? len0 - s * BK : s < sl0 + sl1 ? len1 - (s - sl0) * BK : len2 - (s - sl0 - sl1) * BK); };
    const unsigned lds_base = uniform((int)(size_t)(lds_void_ptr)&lds[0][0]);
    constexpr unsigned kStageBytes = (TA::ELEMS + TB::ELEMS) * 2;
    auto locate = [&](int s, int stage) __attribute__((always_inline)) {
        const int left = left_of(s);
        int lda = lda0, ldb = ldb0;
        const bf16_t* Ap = A0;
        const bf16_t* Bp = B0;
        if (s >= sl0) {
            s -= sl0;
            Ap = A1; Bp = B1; lda = lda1; ldb = ldb1;
            if (s >= sl1) {
                s -= sl1;
                Ap = A2; Bp = B2; lda = lda2; ldb = ldb2;
            }
        }
        const int k0 = s * BK;
        SlabSource src;
        src.a0 = A_KC ? Ap + (long long)m0 * lda + k0 : Ap + (long long)k0 * lda + m0;
        src.b0 = B_KC ? Bp + (long long)n0 * ldb + k0 : Bp + (long long)k0 * ldb + n0;
        set_offsets(lda, ldb, left);
        const unsigned at = (unsigned)uniform((int)(lds_base + (unsigned)stage * kStageBytes));
        src.lds_a = at + (unsigned)wave * (TA::LOADS * 1024);
        src.lds_b = at + TA::ELEMS * 2 + (unsigned)wave * (TB::LOADS * 1024);
        return src;
    };
    // loads h_lo..h_hi-1 of the NLOADS this wave issues per slab
    auto issue = [&](const SlabSource& src, auto h_lo_c, auto h_hi_c) __attribute__((always_inline)) {
        constexpr int h_lo = decltype(h_lo_c)::value, h_hi = decltype(h_hi_c)::value;
        static_for<h_hi - h_lo>([&](auto h_c) {
            constexpr int h = h_lo + decltype(h_c)::value;
            if constexpr (h < TA::LOADS) load_to_lds_16_at<h * 1024>(src.a0, a_off[h], src.lds_a);
            else load_to_lds_16_at<(h - TA::LOADS) * 1024>(src.b0, b_off[h - TA::LOADS], src.lds_b);
        });
    };
    using I0 = std::integral_constant<int, 0>;
    using IN = std::integral_constant<int, NLOADS>;
    if (nk > 0) issue(locate(0, 0), I0{}, IN{});
    if (nk > 1) issue(locate(1, 1), I0{}, IN{});
    int stage = 0;
    // One slab.  REFILL: the loads of slab kt+2 are issued, spread over the contraction steps behind each step's MFMAs, into the stage
    // that held slab kt-1.  TAIL: only `left` of its contraction indices exist.
    auto slab = [&](int kt, int left, auto refill_c, auto tail_c) __attribute__((always_inline)) {
        constexpr bool REFILL = decltype(refill_c)::value, TAIL = decltype(tail_c)::value;
        // slab kt has landed when at most the loads of slab kt+1 are outstanding
        if (REFILL || kt + 1 < nk) wait_loads_but<NLOADS>();
        else wait_loads_but<0>();
        barrier_no_fence();  // slab kt is complete in LDS; every wave is done with slab kt-1
        __builtin_amdgcn_s_setprio(2);
        SlabSource next;
        if (REFILL) next = locate(kt + 2, stage == 0 ? 2 : stage - 1);
        const bf16_t* As = lds[stage];
        const bf16_t* Bs = lds[stage] + TA::ELEMS;
        // operand registers of step st+1 are read from LDS while the MFMAs of step st run
        bf16x8 a[2][TM], b[2][TN];
        auto read = [&](int st, int set) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TM; i++) a[set][i] = TA::fragment(As, wm * WM + i * 32, st * 16, lane);
#pragma unroll
            for (int j = 0; j < TN; j++) b[set][j] = TB::fragment(Bs, wn * WN + j * 32, st * 16, lane);
            if constexpr (TAIL) {
                const int k = st * 16 + 8 * (lane >> 5);
#pragma unroll
                for (int i = 0; i < TM; i++) a[set][i] = zero_from(a[set][i], k, left);
#pragma unroll
                for (int j = 0; j < TN; j++) b[set][j] = zero_from(b[set][j], k, left);
            }
        };
        read(0, 0);
        constexpr int kReadsStep = TM * (A_KC ? 1 : 2) + TN * (B_KC ? 1 : 2);
        if (!TAIL) __builtin_amdgcn_sched_group_barrier(0x100, kReadsStep, 0);
        static_for<KSTEPS>([&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
            if (TAIL && !REFILL && st * 16 >= left) return;  // nothing left of the last slab
            if (st + 1 < KSTEPS) read(st + 1, (st + 1) & 1);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st & 1][i], b[st & 1][j], acc[i][j], 0, 0, 0);
            if (REFILL) issue(next, std::integral_constant<int, st * NLOADS / KSTEPS>{}, std::integral_constant<int, (st + 1) * NLOADS / KSTEPS>{});
            // pin the order: each MFMA of this step is followed by its share of the next step's operand reads
            if (!TAIL) {
                if (st + 1 < KSTEPS) {
                    static_for<TM * TN>([&](auto m_c) {
                        constexpr int mi = decltype(m_c)::value;
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        constexpr int r_lo = mi * kReadsStep / (TM * TN), r_hi = (mi + 1) * kReadsStep / (TM * TN);
                        if (r_hi > r_lo) __builtin_amdgcn_sched_group_barrier(0x100, r_hi - r_lo, 0);
                    });
                } else {
                    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
                }
            }
        });
        __builtin_amdgcn_s_setprio(0);
        stage = stage == 2 ? 0 : stage + 1;
    };
    for (int kt = 0; kt < nk;) {
        for (; kt + 2 < nk && left_of(kt) == BK; kt++) slab(kt, BK, std::true_type{}, std::false_type{});
        if (kt >= nk) break;
        const int left = left_of(kt);
        if (kt + 2 < nk) slab(kt, left, std::true_type{}, std::true_type{});
        else if (left == BK) slab(kt, left, std::false_type{}, std::false_type{});
        else slab(kt, left, std::false_type{}, std::true_type{});
        kt++;
    }
    barrier_no_fence();  // the epilogue reuses the operand LDS

    TC* C = static_cast<TC*>(g.C) + (long long)bz * g.sC;
    const TC* Rsrc = g.R ? static_cast<const TC*>(g.R) + (long long)bz * g.sC : C;
    gemm_store_tile<BM, BN, WGM, WGN, true, sizeof(lds), TC>(g, acc, reinterpret_cast<float*>(&lds[0][0]), C, Rsrc, g.accumulate || g.R != nullptr, bz, split, part, m0,
                                                             n0, wave, wm, wn, lane);
}

template <int BM, typename TC>
void launch_edge(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc) {
    if (a_kc && b_kc) gemm_edge_kernel<BM, true, true, TC><<<(unsigned)g.blocks, 512, 0, ctx->stream>>>(g);
    else if (a_kc) gemm_edge_kernel<BM, true, false, TC><<<(unsigned)g.blocks, 512, 0, ctx->stream>>>(g);
    else if (b_kc) gemm_edge_kernel<BM, false, true, TC><<<(unsigned)g.blocks, 512, 0, ctx->stream>>>(g);
    else gemm_edge_kernel<BM, false, false, TC><<<(unsigned)g.blocks, 512, 0, ctx->stream>>>(g);
}

}  // namespace

void eisen_gemm_launch_edge(eisen_ctx* ctx, GemmArgs g, int tile_rows, bool a_kc, bool b_kc, int batch, int dtype_c) {
    g.blocks = (int)eisen_ceil_div(g.M, tile_rows) * (int)eisen_ceil_div(g.N, 128) * batch * (g.split > 1 ? g.split : 1);
    if (tile_rows == 256 && dtype_c == EISEN_BF16) launch_edge<256, bf16_t>(ctx, g, a_kc, b_kc);
    else if (tile_rows == 256) launch_edge<256, float>(ctx, g, a_kc, b_kc);
    else if (dtype_c == EISEN_BF16) launch_edge<128, bf16_t>(ctx, g, a_kc, b_kc);
    else launch_edge<128, float>(ctx, g, a_kc, b_kc);
}

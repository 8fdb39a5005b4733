// f32 GEMM on the bf16 matrix cores: C[M,N] (+)= op(A) * op(B) in tiles whose contraction is dealt to the waves of the workgroup, as
// in gemm_sliced.hip, for f32 operands whose rows start on 16-byte boundaries (others: gemm_f32.hip).
//
// Precision.  An f32 value is the exact sum of three bf16 values (8 bits each, round to nearest) once it is multiplied by 2^23, which lifts
// the last place of the smallest f32 values into bf16's range.  Of the nine products of two such sums six are formed, all in one f32
// accumulator; two of the others reach 2^-25 of a product each, so that what is left out stays below 2^-23.9 of it, where an f32
// multiply-add rounds at 2^-24 of its sum.  An MFMA of 16 contraction indices rounds its accumulator once, so 16 indices cost 6 roundings
// where the f32 MFMAs take 16; what the bf16 MFMAs cut off leans towards minus infinity, and every other wave therefore adds up the
// negative of its share.  A slice's small products come first, when there is little to round off (in turn per 16 indices: K = 32 6.9e-8, of
// positive operands 5.6e-8, which is more than the f32 MFMAs).
// Error against float64 relative to the result (2-norm), f32 MFMAs / here: N(0, 1) operands, K = 4 4.0e-8 / 3.2e-8, 32 6.8e-8 / 3.8e-8, 64
// 8.4e-8 / 4.6e-8, 256 1.5e-7 / 6.8e-8, 1000 2.9e-7 / 1.6e-7, 4096 2.9e-7 / 1.7e-7; positive operands 32 4.5e-8 / 3.5e-8, 256 6.9e-8 / 4.8e-8,
// 4096 7.3e-8 / 4.9e-8; operands of 2^-140 at K = 256 1.5e-7 / 6.5e-8 (without the factor 1.6e-7 at 2^-112, 3.5e-5 at 2^-120, nothing left
// at 2^-140; it costs two vector instructions per pair of elements less those of the signs that it carries, 0 to 5 % of a product's time).
// A value that is not finite, a factor from 2^104 on, which rounds to infinity in bf16 then, or a sum from 2^81 on makes some output of its
// tile not finite: such a tile is computed again with f32 MFMAs (once more its time), so infinities and NaN come out as they do there.
//
// What bounds it: the f32 MFMAs need 1024 cycles per SIMD for a 64 x 64 x 32 slice, six bf16 products 384, beside 400 vector instructions of 4
// cycles per wave that split the operands; the units overlap only in part (4096 x 256 x 8192, before the factor: 64 us with the loads alone, 81 with split
// and MFMAs alone, 99 together, 162 on the f32 MFMAs).  A wave owns the whole tile of its slice, so every element is split once per tile, in
// registers.  us, gemm_f32.hip / here, operands from memory: 4096 x 256 x 256 10.9 / 8.8, 4096 x 1024 x 256 31.2 / 24.4, 4096 x 256 x 8192 NT 164 / 114, 2048^3
// 157 / 111, weight gradients 256 x 1024 x 4096 30.0 / 23.3, 8192 x 256 x 4096 157 / 114; 32 x 32 tiles: 64 x 64 x 64 5.0 / 4.3, 200 x 256 x 256 7.0 / 5.2, 512 x 384 x 1024
// 14.2 / 8.6, 288 x 768 x 1352 15.9 / 11.2, 1352 x 288 x 1536 NT 23.7 / 18.5.
#include "gemm_common.cuh"

namespace {

constexpr int FK = 32;  // depth of a slice

enum class Kind { kPlain, kSegments, kGroup, kSwiglu, kLayers };
struct NoLayers {};

// integer divisions leave values that are the same in every lane in vector registers
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// One operand of a slice in the LDS as memory has it: stored along the contraction, T rows (m or n) of 128 bytes; stored the
// other way round, 32 rows (k) of 4 T bytes.
template <int T, bool KC>
struct F32SliceTile {
    static constexpr int CPR = KC ? 8 : T / 4, ROWS = 64 / CPR, LOADS = T / 8;  // 16-byte chunks per row, rows per load, loads
    // Which row and chunk of the operand stand at a place in the LDS.  Along the contraction the chunks are permuted by row: 16 rows at
    // one chunk fall into 16 different 16-byte slots of the 64 banks.  The other way round a wave reads rows 8 apart at a time: they use
    // different halves of the banks.
    static __device__ __forceinline__ int row_at(int row) { return !KC && T == 32 ? row ^ (row >> 3 & 1) : row; }
    static __device__ __forceinline__ int chunk_at(int row, int chunk) { return KC ? chunk ^ lds_swz<128>(row) : T == 64 ? chunk ^ (row & 8) : chunk; }
    // row_last, chunk_last: the last ones that exist
    static __device__ __forceinline__ void load(const float* base, int ld, unsigned tile, int row_last, int chunk_last, int lane) {
        const int row = lane / CPR;
        if (row_last >= ROWS * LOADS - 1 && chunk_last >= CPR - 1) {
            unsigned off[2];  // the permutations repeat every 16 rows
#pragma unroll
            for (int odd = 0; odd < 2; odd++) off[odd] = (unsigned)((row_at(row + 8 * odd) - 8 * odd) * ld + chunk_at(row + 8 * odd, lane % CPR) * 4) * 4u;
            static_for<LOADS>([&](auto i_c) {
                constexpr int i = decltype(i_c)::value;
                load_to_lds_16_at<i * 1024>(base + (long long)i * ROWS * ld, off[(i * ROWS >> 3) & 1], tile);
            });
        } else {
            static_for<LOADS>([&](auto i_c) {
                constexpr int i = decltype(i_c)::value;
                const int r = row + i * ROWS;
                load_to_lds_16_at<i * 1024>(base, (unsigned)(min(row_at(r), row_last) * ld + min(chunk_at(r, lane % CPR), chunk_last) * 4) * 4u, tile);
            });
        }
    }
    // The same for T/2 columns each of two operands [K][N] side by side: the first half of a row's chunks is the first one's.  The operands start `first` and
    // `second` bytes behind base (32-bit offsets: a 64-bit address per lane and load would cost the vector unit, which bounds the kernel).
    static __device__ __forceinline__ void load_two(const float* base, unsigned first, unsigned second, int ld, unsigned tile, int row_last, int chunk_last, int lane) {
        static_assert(!KC, "columns side by side");
        constexpr int HALF = CPR / 2;
        const int row = lane / CPR;
        auto at = [&](int chunk, int last) __attribute__((always_inline)) { return (unsigned)min(chunk % HALF, last) * 16u + (chunk < HALF ? first : second); };
        if (row_last >= ROWS * LOADS - 1 && chunk_last >= HALF - 1) {
            unsigned off[2];
#pragma unroll
            for (int odd = 0; odd < 2; odd++) off[odd] = (unsigned)((row_at(row + 8 * odd) - 8 * odd) * ld) * 4u + at(chunk_at(row + 8 * odd, lane % CPR), HALF - 1);
            static_for<LOADS>([&](auto i_c) {
                constexpr int i = decltype(i_c)::value;
                load_to_lds_16_at<i * 1024>(base + (long long)i * ROWS * ld, off[(i * ROWS >> 3) & 1], tile);
            });
        } else {
            static_for<LOADS>([&](auto i_c) {
                constexpr int i = decltype(i_c)::value;
                const int r = row + i * ROWS;
                load_to_lds_16_at<i * 1024>(base, (unsigned)(min(row_at(r), row_last) * ld) * 4u + at(chunk_at(r, lane % CPR), chunk_last), tile);
            });
        }
    }
    // contraction indices ks + 8 (lane / 32) + 0..7 of operand row row0 + lane % 32
    static __device__ __forceinline__ void fragment(const char* tile, int row0, int ks, int lane, float (&f)[8]) {
        const int r = row0 + (lane & 31), gh = lane >> 5;
        if constexpr (KC) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const float4 v = *reinterpret_cast<const float4*>(tile + r * 128 + (chunk_at(r, ks / 4 + 2 * gh + q) << 4));
                f[4 * q] = v.x; f[4 * q + 1] = v.y; f[4 * q + 2] = v.z; f[4 * q + 3] = v.w;
            }
        } else if constexpr (T == 64) {
            const float* p = reinterpret_cast<const float*>(tile) + (ks + 8 * gh) * 64 + (r ^ (gh * 32));
#pragma unroll
            for (int j = 0; j < 8; j++) f[j] = p[j * 64];
        } else {
            const float* even = reinterpret_cast<const float*>(tile) + (ks + 9 * gh) * 32 + r;
            const float* odd = reinterpret_cast<const float*>(tile) + (ks + 7 * gh) * 32 + r;
#pragma unroll
            for (int j = 0; j < 8; j++) f[j] = (j & 1 ? odd : even)[j * 32];
        }
    }
};

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Operands are multiplied by a power of two before they are split: the last place of the smallest f32 value (2^-149) is then bf16's smallest
// normal one, so that every part of every value is there.
constexpr float kScale = 0x1p23f;
constexpr float kUnscale = 0x1p-46f;  // of a product of two

// scale * x = hi + mid + lo, exactly (8 bits each, rounded to nearest) where scale * x rounds to a finite bf16; scale: a power of two or its negative
__device__ __forceinline__ void split_bf16(const float (&x)[8], float scale, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
    u32x4 h, m, l;
    auto pack = [](float x0, float x1) { return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x0, x1}, bf16x2)); };
    auto low = [](unsigned u) { return __builtin_bit_cast(float, u << 16); };
    auto high = [](unsigned u) { return __builtin_bit_cast(float, u & 0xffff0000u); };
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float x0 = x[2 * e] * scale, x1 = x[2 * e + 1] * scale;
        h[e] = pack(x0, x1);
        const float r0 = x0 - low(h[e]), r1 = x1 - high(h[e]);
        m[e] = pack(r0, r1);
        l[e] = pack(r0 - low(m[e]), r1 - high(m[e]));
    }
    hi = __builtin_bit_cast(bf16x8, h);
    mid = __builtin_bit_cast(bf16x8, m);
    lo = __builtin_bit_cast(bf16x8, l);
}

template <int W, int FT, bool A_KC, bool B_KC, Kind KIND>
__global__ __launch_bounds__(64 * W, 2) void gemm_f32_sliced_kernel(GemmArgs g, std::conditional_t<KIND == Kind::kLayers, DwArgs, NoLayers> layers) {
    using TA = F32SliceTile<FT, A_KC>;
    using TB = F32SliceTile<FT, B_KC>;
    constexpr int TM = FT / 32, kOperandBytes = FT * FK * 4;
    constexpr int COLS = KIND == Kind::kSwiglu ? FT / 2 : FT;  // columns of each product
    static_assert(2 * kOperandBytes >= FT * FT * (int)sizeof(float), "a wave's partial tile takes the place of its slice");
    __shared__ __attribute__((aligned(1024))) char lds[W][2 * kOperandBytes];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int split = g.split > 1 ? g.split : 1;
    constexpr bool kRope = KIND == Kind::kGroup && A_KC && !B_KC;  // (the rotary epilogue: of X W)
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
                if constexpr (kRope) member = q;
                first = g.grp_tile_end[q - 1];
                partial_off = g.grp_partial_off[q];
                g.A = g.grp_A[q]; g.B = g.grp_B[q]; g.C = g.grp_C[q]; g.N = g.grp_N[q];
            }
        if (split > 1) g.partial += partial_off;
        const int n_tiles = (g.N + FT - 1) / FT;
        mt = (t - first) / n_tiles;
        nt = (t - first) % n_tiles;
        g.ldc = g.N;
        if (!B_KC) g.ldb = g.N;
    } else if constexpr (KIND == Kind::kLayers) {  // every lane looks at one product
        int t = xcd_contiguous_id(blockIdx.x, layers.tiles);
        const int p = __popcll(__ballot(lane < layers.n && t >= layers.tile_end[lane]));
        const DwProduct& pr = layers.p[p];
        if (p > 0) t -= layers.tile_end[p - 1];
        g.A = pr.A; g.B = pr.B; g.C = pr.C; g.M = pr.M; g.N = pr.N;
        g.lda = g.M; g.ldb = g.ldc = g.N;
        g.accumulate = pr.accumulate;
        zz = 0;
        block_tile<4, 8>(t, (g.M + FT - 1) / FT, (g.N + FT - 1) / FT, mt, nt);
    } else {
        const int gx = (g.N + COLS - 1) / COLS, gy = (g.M + FT - 1) / FT;
        const int lin = xcd_contiguous_id(blockIdx.x, g.blocks);
        zz = uniform(lin / (gx * gy));
        block_tile<4, 8>(lin - zz * (gx * gy), gy, gx, mt, nt);
    }
    const int m0 = uniform(mt * FT), n0 = uniform(nt * COLS);
    const int bz = uniform(zz / split), part = uniform(zz % split);
    const float* A = static_cast<const float*>(g.A) + (KIND == Kind::kSwiglu ? 0 : (long long)bz * g.sA);
    const float* B = static_cast<const float*>(g.B) + (KIND == Kind::kSwiglu ? 0 : (long long)bz * g.sB);

    // Slices of the contraction: segment by segment, each with a last slice of its own.  This workgroup's are [s_lo, s_hi).
    constexpr bool SEG = KIND == Kind::kSegments;
    const int len0 = SEG ? g.seg_end[0] : g.K;
    const int sl0 = (len0 + FK - 1) / FK;
    const int len1 = !SEG ? 0 : g.nseg > 2 ? g.seg_end[1] - g.seg_end[0] : g.K - g.seg_end[0], sl1 = (len1 + FK - 1) / FK;
    const int len2 = SEG && g.nseg > 2 ? g.K - g.seg_end[1] : 0, sl2 = (len2 + FK - 1) / FK;
    const float *A1 = nullptr, *A2 = nullptr, *B1 = nullptr, *B2 = nullptr;
    int lda1 = 0, lda2 = 0, ldb1 = 0, ldb2 = 0;
    const int lda0 = g.lda, ldb0 = g.ldb;
    if constexpr (SEG) {
        A1 = static_cast<const float*>(g.A_seg[0]); A2 = static_cast<const float*>(g.A_seg[1]);
        B1 = static_cast<const float*>(g.B_seg[0]); B2 = static_cast<const float*>(g.B_seg[1]);
        lda1 = g.lda_seg[0]; lda2 = g.lda_seg[1];
        ldb1 = g.ldb_seg[0]; ldb2 = g.ldb_seg[1];
    }
    const int s_lo = part * (g.k_part / FK), s_hi = split > 1 ? min(sl0, s_lo + g.k_part / FK) : sl0 + sl1 + sl2;
    const int n_mine = s_hi - s_lo > wave ? (s_hi - s_lo - wave + W - 1) / W : 0;
    const int n_parts = min(W, s_hi - s_lo);  // waves with something to add

    char* As = lds[wave];
    char* Bs = As + kOperandBytes;
    const int m_last = g.M - 1 - m0, n_last = g.N - 1 - n0;  // last row of the tile that exists
    const unsigned lds_a = uniform((int)(size_t)(lds_void_ptr)As), lds_b = lds_a + kOperandBytes;  // their LDS addresses
    // the loads of this wave's i-th slice; returns how many of its contraction indices exist
    auto issue = [&](int i) __attribute__((always_inline)) -> int {
        int s = s_lo + wave + i * W, lda = lda0, ldb = ldb0, len = len0;
        const float* Ap = A;
        const float* Bp = B;
        if (SEG && s >= sl0) {
            s -= sl0;
            Ap = A1; Bp = B1; lda = lda1; ldb = ldb1; len = len1;
            if (s >= sl1) {
                s -= sl1;
                Ap = A2; Bp = B2; lda = lda2; ldb = ldb2; len = len2;
            }
        }
        const int k0 = s * FK, left = len - k0;
        TA::load(A_KC ? Ap + (long long)m0 * lda + k0 : Ap + (long long)k0 * lda + m0, lda, lds_a, A_KC ? m_last : left - 1, (A_KC ? left - 1 : m_last) / 4, lane);
        if constexpr (KIND == Kind::kSwiglu)
            TB::load_two(Bp + (long long)k0 * ldb + n0, (unsigned)g.sA, (unsigned)g.sB, ldb, lds_b, left - 1, n_last / 4, lane);
        else
            TB::load(B_KC ? Bp + (long long)n0 * ldb + k0 : Bp + (long long)k0 * ldb + n0, ldb, lds_b, B_KC ? n_last : left - 1, (B_KC ? left - 1 : n_last) / 4, lane);
        return min(left, FK);
    };

    // groups of eight columns: of the tile, per thread; with the SwiGLU a thread has a group of the gate and the same one of up
    constexpr int GROUPS = FT * FT / 8, HALF = FT / 16, PASSES = KIND == Kind::kSwiglu ? 2 : (GROUPS + 64 * W - 1) / (64 * W);
    auto has_group = [&](int ps) { return KIND == Kind::kSwiglu ? tid < GROUPS / 2 : GROUPS % (64 * W) == 0 || ps * 64 * W + tid < GROUPS; };
    auto group_row = [&](int ps) { return KIND == Kind::kSwiglu ? tid / HALF : (ps * 64 * W + tid) / (FT / 8); };
    auto group_of = [&](int ps) { return KIND == Kind::kSwiglu ? tid % HALF + ps * HALF : (ps * 64 * W + tid) % (FT / 8); };
    float* C = static_cast<float*>(g.C) + (long long)bz * g.sC;
    const float* Rsrc = g.R ? static_cast<const float*>(g.R) + (long long)bz * g.sC : C;
    float* P = gemm_partial<float>(g, bz, split, part);
    const bool add_old = (g.accumulate || g.R != nullptr) && !P && !g.gate;

    f32x16 acc[TM][TM];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
    };
    // contraction indices 16 st .. 16 st + 15 of the slice in the LDS
    auto read = [&](int st, float (&a)[TM][8], float (&b)[TM][8]) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < TM; h++) {
            TA::fragment(As, h * 32, st * 16, lane, a[h]);
            TB::fragment(Bs, h * 32, st * 16, lane, b[h]);
        }
    };
    // zeros from the slice's index `now` on
    auto cut = [&](int st, int now, float (&a)[TM][8], float (&b)[TM][8]) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < TM; h++)
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (st * 16 + 8 * (lane >> 5) + e >= now) a[h][e] = b[h][e] = 0.f;
    };
    // The waves' tiles, each in the place of its (now idle) slice, rows 4 apart (the two halves of a wave) in different halves of the
    // banks; then their sum, eight columns of a row per thread.
    auto place = [](int r, int n) { return FT == 64 ? r * 64 + (n ^ ((r >> 2 & 1) * 32)) : (r ^ (r >> 2 & 1)) * 32 + n; };
    float val[PASSES][8];
    auto meet = [&](float odd, float unscale) __attribute__((always_inline)) -> int {
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
        int bad = 0;
        static_for<PASSES>([&](auto ps_c) {
            constexpr int ps = decltype(ps_c)::value;
            const int r = group_row(ps), cg = group_of(ps);
#pragma unroll
            for (int e = 0; e < 8; e++) val[ps][e] = 0.f;
            if (!has_group(ps)) return;
            const float* src = reinterpret_cast<const float*>(lds[0]) + place(r, cg * 8);
            for (int w = 0; w < n_parts; w++) {  // in wave order
                const float4 lo = *reinterpret_cast<const float4*>(src + w * (kOperandBytes / 2)), hi = *reinterpret_cast<const float4*>(src + w * (kOperandBytes / 2) + 4);
                const float sg = w & 1 ? odd : 1.f;
                val[ps][0] += sg * lo.x; val[ps][1] += sg * lo.y; val[ps][2] += sg * lo.z; val[ps][3] += sg * lo.w;
                val[ps][4] += sg * hi.x; val[ps][5] += sg * hi.y; val[ps][6] += sg * hi.z; val[ps][7] += sg * hi.w;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) val[ps][e] *= unscale;
            if (m0 + r < g.M)
#pragma unroll
                for (int e = 0; e < 8; e++) bad |= n0 + cg * 8 % COLS + e < g.N && !(fabsf(val[ps][e]) < INFINITY);
        });
        return bad;
    };

    if (W == 8 ? wave >= 4 : (blockIdx.x >> 8) & 1) __builtin_amdgcn_s_setprio(2);
    // The bf16 MFMAs cut the bits below their accumulator's last place off towards minus infinity; every other wave adds up the negative of
    // its share, so that what is cut off cancels.
    const float scale_a = wave & 1 ? -kScale : kScale;
    int left = 0;
    if (n_mine > 0) left = issue(0);
    clear();
    // kLayers: four waves take whole contractions, where other launches give eight waves a part each.  The sums of two slices are added to a total, so that no accumulator
    // rounds a longer one; where those launches leave a wave a slice or few (contractions of at most eight slices, products of fewer than 64 tiles of 64 x 64, which
    // they split), every slice by itself, and what the addition to the total rounds away opens the next slice's sum.  Error against float64, each slice / two slices /
    // a launch of its own: 64 x 64 x 256 6.0e-8 / 1.0e-7 / 6.6e-8, 96 x 256 x 1351 6.3e-8 / 1.1e-7 / 9.0e-8, 256 x 256 x 4096 6.3e-8 / 1.3e-7 / 1.7e-7, 64 x 64 x 16384
    // 6.3e-8 / 1.8e-7 / 1.5e-7, 256 x 1024 x 4096 6.2e-8 / 1.3e-7 / 1.7e-7 (all of a wave's slices in one accumulator 4.9e-7).  us, the products of the ~14 M model's layers
    // over 4096 tokens, each slice everywhere / this / two slices everywhere 492 / 455 / 438, in launches of their own 832.
    f32x16 total[KIND == Kind::kLayers ? TM : 1][KIND == Kind::kLayers ? TM : 1] = {};
    auto add_to_total = [&](auto carry_c) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < TM; p++)
#pragma unroll
            for (int q = 0; q < TM; q++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float sum = total[p][q][v] + acc[p][q][v];
                    acc[p][q][v] = decltype(carry_c)::value ? acc[p][q][v] - (sum - total[p][q][v]) : 0.f;
                    total[p][q][v] = sum;
                }
    };
    auto slice = [&](int i) __attribute__((always_inline)) {
        wait_loads_but<0>();
        float a[2][TM][8], b[2][TM][8];
        read(0, a[0], b[0]);
        read(1, a[1], b[1]);
        const int now = left;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slice is in registers: the next one may overwrite it
        if (i + 1 < n_mine) left = issue(i + 1);
        if (now < FK) {
            cut(0, now, a[0], b[0]);
            cut(1, now, a[1], b[1]);
        }
        // Splitting an operand's 32 rows x 16 indices takes 52 vector instructions of 4 cycles, the six products of a 32 x 32 x 16 block six
        // MFMAs of 32: each block's MFMAs go out with the vector instructions that split what the block after next needs between
        // them.  (Split first, then multiplied, the waves of a SIMD do both in step and neither unit covers the other.)
        bf16x8 ap[2][TM][3], bp[2][TM][3];
        auto split_a = [&](auto st_c, auto h_c) { constexpr int st = decltype(st_c)::value, h = decltype(h_c)::value; split_bf16(a[st][h], scale_a, ap[st][h][0], ap[st][h][1], ap[st][h][2]); };
        auto split_b = [&](auto st_c, auto h_c) { constexpr int st = decltype(st_c)::value, h = decltype(h_c)::value; split_bf16(b[st][h], kScale, bp[st][h][0], bp[st][h][1], bp[st][h][2]); };
        // The products of a step's parts, small ones first; those of the first parts, whose sums round at the size of the result, wait
        // for the second step's small ones.
        auto block = [&](auto st_c, auto p_c, auto q_c, auto with_split) {
            constexpr int st = decltype(st_c)::value, p = decltype(p_c)::value, q = decltype(q_c)::value;
            constexpr int order[5][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
            static_for<5>([&](auto o_c) {
                constexpr int o = decltype(o_c)::value;
                acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ap[st][p][order[o][0]], bp[st][q][order[o][1]], acc[p][q], 0, 0, 0);
            });
            if constexpr (st == 1)
                static_for<2>([&](auto o_c) { constexpr int o = decltype(o_c)::value; acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ap[o][p][0], bp[o][q][0], acc[p][q], 0, 0, 0); });
            constexpr int mfmas = st == 1 ? 7 : 5;
            if constexpr (decltype(with_split)::value) {
                static_for<mfmas>([&](auto) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, FT == 32 ? 21 : st == 1 ? 8 : 11, 0);
                });
            } else {
                __builtin_amdgcn_sched_group_barrier(0x008, mfmas, 0);
            }
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using Yes = std::true_type;
        using No = std::false_type;
        split_a(I0{}, I0{});
        split_b(I0{}, I0{});
        __builtin_amdgcn_sched_group_barrier(0x002, 104, 0);
        if constexpr (FT == 64) {
            split_a(I0{}, I1{}); block(I0{}, I0{}, I0{}, Yes{});
            split_b(I0{}, I1{}); block(I0{}, I1{}, I0{}, Yes{});
            split_a(I1{}, I0{}); block(I0{}, I0{}, I1{}, Yes{});
            split_b(I1{}, I0{}); block(I0{}, I1{}, I1{}, Yes{});
            split_a(I1{}, I1{}); block(I1{}, I0{}, I0{}, Yes{});
            split_b(I1{}, I1{}); block(I1{}, I1{}, I0{}, Yes{});
            block(I1{}, I0{}, I1{}, No{});
            block(I1{}, I1{}, I1{}, No{});
        } else {
            split_a(I1{}, I0{});
            split_b(I1{}, I0{});
            block(I0{}, I0{}, I0{}, Yes{});
            block(I1{}, I0{}, I0{}, No{});
        }
    };
    if constexpr (KIND == Kind::kLayers) {
        if (g.K <= 8 * FK || ((g.M + 63) / 64) * ((g.N + 63) / 64) < 64) {
            for (int i = 0; i < n_mine; i++) {
                if (i > 0) add_to_total(std::true_type{});
                slice(i);
            }
        } else {
            for (int i = 0; i < n_mine; i++) {
                if (i > 0 && i % 2 == 0) add_to_total(std::false_type{});
                slice(i);
            }
        }
        add_to_total(std::false_type{});
#pragma unroll
        for (int p = 0; p < TM; p++)
#pragma unroll
            for (int q = 0; q < TM; q++) acc[p][q] = total[p][q];
    } else {
        for (int i = 0; i < n_mine; i++) slice(i);
    }
    const int bad = meet(-1.f, kUnscale);
    if (__syncthreads_or(bad)) {  // something that is not finite: once more in f32
        clear();
        for (int i = 0; i < n_mine; i++) {
            const int now = issue(i);
            wait_loads_but<0>();
#pragma unroll
            for (int st = 0; st < 2; st++) {
                float a[TM][8], b[TM][8];
                read(st, a, b);
                cut(st, now, a, b);
#pragma unroll
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int p = 0; p < TM; p++)
#pragma unroll
                        for (int q = 0; q < TM; q++) acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[p][e], b[q][e], acc[p][q], 0, 0, 0);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        (void)meet(1.f, 1.f);
    }
    if constexpr (KIND == Kind::kSwiglu) {  // N is a multiple of 8 and the results start on 16-byte boundaries
        const int m = m0 + group_row(0), n = n0 + group_of(0) * 8;
        if (!has_group(0) || m >= g.M || n >= g.N) return;
        float h[8];
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = val[0][e] * (1.0f / (1.0f + __expf(-val[0][e]))) * val[1][e];
        const long long at = (long long)m * g.N + n;
        auto store = [&](void* to, const float (&x)[8]) {
            float4* p = reinterpret_cast<float4*>(static_cast<float*>(to) + at);
            p[0] = make_float4(x[0], x[1], x[2], x[3]);
            p[1] = make_float4(x[4], x[5], x[6], x[7]);
        };
        store(g.C, val[0]);
        store(g.C2, val[1]);
        store(g.grp_C[0], h);
        return;
    }
    static_for<PASSES>([&](auto ps_c) {
        constexpr int ps = decltype(ps_c)::value;
        const int idx = ps * 64 * W + tid, m = m0 + idx / (FT / 8), n = n0 + (idx % (FT / 8)) * 8;
        if (idx >= GROUPS || m >= g.M || n >= g.N) return;
        const long long at = (long long)m * g.ldc + n;
        typename Eight<float>::V first = {}, second = {};
        if (n + 8 <= g.N) {
            if (add_old) first = load_eight(Rsrc + at);
            if (g.gate) {
                first = load_eight(static_cast<const float*>(g.gate) + (long long)bz * g.sC + at);
                second = load_eight(static_cast<const float*>(g.up) + (long long)bz * g.sC + at);
            }
        }
        // (part 0 of a split contraction stands in C as it is: the reduction rotates)
        gemm_store_eight<float, kRope>(g, val[ps], m, n, !kRope ? bz : split > 1 ? g.rope_members : member, C, Rsrc, add_old, P, first, second);
    });
}

template <int W, int FT, Kind KIND>
void launch_f32_sliced(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc) {
    const unsigned grid = (unsigned)g.blocks;
    if (a_kc && b_kc) gemm_f32_sliced_kernel<W, FT, true, true, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g, NoLayers{});
    else if (a_kc) gemm_f32_sliced_kernel<W, FT, true, false, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g, NoLayers{});
    else if (b_kc) gemm_f32_sliced_kernel<W, FT, false, true, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g, NoLayers{});
    else gemm_f32_sliced_kernel<W, FT, false, false, KIND><<<grid, 64 * W, 0, ctx->stream>>>(g, NoLayers{});
}
template <int W, int FT>
void launch_f32_sliced_w(eisen_ctx* ctx, const GemmArgs& g, bool a_kc, bool b_kc) {
    if (g.ngroup > 0) launch_f32_sliced<W, FT, Kind::kGroup>(ctx, g, a_kc, b_kc);
    else if (g.nseg > 1) launch_f32_sliced<W, FT, Kind::kSegments>(ctx, g, a_kc, b_kc);
    else launch_f32_sliced<W, FT, Kind::kPlain>(ctx, g, a_kc, b_kc);
}

}  // namespace

void eisen_gemm_launch_f32_sliced(eisen_ctx* ctx, GemmArgs g, int waves, int tile, bool a_kc, bool b_kc, int batch) {
    const int split = g.split > 1 ? g.split : 1;
    if (g.ngroup > 0) {
        for (int p = g.ngroup; p < kMaxGroup; p++) g.grp_tile_end[p] = g.grp_tile_end[g.ngroup - 1];  // no tile belongs to the missing ones
        g.blocks = g.grp_tile_end[kMaxGroup - 1] * split;
    } else {
        g.blocks = (int)eisen_ceil_div(g.M, tile) * (int)eisen_ceil_div(g.N, tile) * batch * split;
    }
    if (tile == 64 && waves == 8) launch_f32_sliced_w<8, 64>(ctx, g, a_kc, b_kc);
    else if (tile == 64) launch_f32_sliced_w<4, 64>(ctx, g, a_kc, b_kc);
    else if (waves == 8) launch_f32_sliced_w<8, 32>(ctx, g, a_kc, b_kc);
    else launch_f32_sliced_w<4, 32>(ctx, g, a_kc, b_kc);
}

// Weight gradients of many layers (see gemm_dw.hip); rows start on 16-byte boundaries.  Four waves whatever the tile, so that the bits are the same.
void eisen_gemm_launch_f32_dw(eisen_ctx* ctx, const DwArgs& layers, int tile) {
    GemmArgs g{};
    g.K = layers.K;
    if (tile == 64) gemm_f32_sliced_kernel<4, 64, false, false, Kind::kLayers><<<(unsigned)layers.tiles, 256, 0, ctx->stream>>>(g, layers);
    else gemm_f32_sliced_kernel<4, 32, false, false, Kind::kLayers><<<(unsigned)layers.tiles, 256, 0, ctx->stream>>>(g, layers);
}

// G = X Wg, U = X Wu, H = silu(G) * U: A = X [M][K], C = G, C2 = U, grp_C[0] = H; Wg and Wu [K][N] start sA and sB bytes (below 2^31) behind B.
void eisen_gemm_launch_f32_sliced_swiglu(eisen_ctx* ctx, GemmArgs g, int waves, int tile) {
    g.blocks = (int)eisen_ceil_div(g.M, tile) * (int)eisen_ceil_div(g.N, tile / 2);
    const unsigned grid = (unsigned)g.blocks;
    if (tile == 64 && waves == 8) gemm_f32_sliced_kernel<8, 64, true, false, Kind::kSwiglu><<<grid, 512, 0, ctx->stream>>>(g, NoLayers{});
    else if (tile == 64) gemm_f32_sliced_kernel<4, 64, true, false, Kind::kSwiglu><<<grid, 256, 0, ctx->stream>>>(g, NoLayers{});
    else if (waves == 8) gemm_f32_sliced_kernel<8, 32, true, false, Kind::kSwiglu><<<grid, 512, 0, ctx->stream>>>(g, NoLayers{});
    else gemm_f32_sliced_kernel<4, 32, true, false, Kind::kSwiglu><<<grid, 256, 0, ctx->stream>>>(g, NoLayers{});
}

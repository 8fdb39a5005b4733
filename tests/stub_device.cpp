// The graph layer on a stub of the device, for what depends on how far the device has come: buffers are host memory, the main stream's
// work runs at once, the side stream's as late as it may (when something waits for it).  What eisen_hip_side_begin_if_behind answers is
// given on the command line, one digit per call: 1 forked, 0 caught up.
//
// One argument: backward of two products with one weight, Y = (X W) W, in two passes that add up; exit status 0 if the gradients of W and X are
// those of the same graph with the weight gradients on the main stream, bit for bit.  Two arguments: the graph that the first one names.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "../eisen_amd/csrc/host/graph.hpp"

struct eisen_ctx {
    const char* answers = "";
    bool side = false, section = false;
    int forks = 0, inlines = 0, sides = 0;
    std::string order;  // of the products: d(ense), w(eight gradients), each with their number
    std::vector<std::function<void()>> late;  // the side stream
    std::map<void*, size_t> live;            // bytes of every buffer
    size_t bytes() const {
        size_t n = 0;
        for (const auto& b : live) n += b.second;
        return n;
    }
};

static float widen(uint16_t h) {
    const uint32_t u = (uint32_t)h << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}
static uint16_t narrow(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return (uint16_t)((u + 0x7fff + (u >> 16 & 1)) >> 16);
}
static float get(const void* p, size_t i, int dtype) { return dtype == EISEN_BF16 ? widen(((const uint16_t*)p)[i]) : ((const float*)p)[i]; }
static void put(void* p, size_t i, int dtype, float v) {
    if (dtype == EISEN_BF16) ((uint16_t*)p)[i] = narrow(v);
    else ((float*)p)[i] = v;
}
static int give(eisen_ctx* ctx, std::function<void()> work) {
    if (ctx->side) ctx->late.push_back(std::move(work));
    else work();
    return 0;
}

extern "C" {
const char* eisen_hip_last_error(eisen_ctx*) { return "refused by the stub"; }
int eisen_hip_malloc_zeroed(eisen_ctx* ctx, size_t bytes, void** out) {
    if (!(*out = std::calloc(bytes + 16, 1))) return -1;
    ctx->live[*out] = bytes;
    return 0;
}
int eisen_hip_malloc(eisen_ctx* ctx, size_t bytes, void** out) { return eisen_hip_malloc_zeroed(ctx, bytes, out); }
int eisen_hip_free(eisen_ctx* ctx, void* p) {
    if (ctx->live.erase(p) != 1) return -1;
    return give(ctx, [=] { std::free(p); });
}
int eisen_hip_memset_zero(eisen_ctx* ctx, void* p, size_t bytes) { return give(ctx, [=] { std::memset(p, 0, bytes); }); }
int eisen_hip_htod(eisen_ctx*, void* d, const void* s, size_t bytes) { return std::memcpy(d, s, bytes), 0; }
int eisen_hip_dtod(eisen_ctx* ctx, void* d, const void* s, size_t bytes) { return give(ctx, [=] { std::memmove(d, s, bytes); }); }
int eisen_hip_fill(eisen_ctx* ctx, void* p, int dtype, float v, size_t n) {
    return give(ctx, [=] { for (size_t i = 0; i < n; i++) put(p, i, dtype, v); });
}
int eisen_hip_cast(eisen_ctx* ctx, const void* s, int from, void* d, int to, size_t n) {
    return give(ctx, [=] { for (size_t i = 0; i < n; i++) put(d, i, to, get(s, i, from)); });
}
int eisen_hip_gemm(eisen_ctx* ctx, const void* A, const void* B, void* C, int dtype_ab, int dtype_c, int ta, int tb, size_t M, size_t N, size_t K, int accumulate) {
    ctx->order += 'd';
    return give(ctx, [=] {
        std::vector<float> b(K * N), sum(N);
        for (size_t k = 0; k < K; k++)
            for (size_t n = 0; n < N; n++) b[k * N + n] = get(B, tb ? n * K + k : k * N + n, dtype_ab);
        for (size_t m = 0; m < M; m++) {
            for (size_t n = 0; n < N; n++) sum[n] = accumulate ? get(C, m * N + n, dtype_c) : 0.f;
            for (size_t k = 0; k < K; k++) {
                const float a = get(A, ta ? k * M + m : m * K + k, dtype_ab);
                for (size_t n = 0; n < N; n++) sum[n] += a * b[k * N + n];
            }
            for (size_t n = 0; n < N; n++) put(C, m * N + n, dtype_c, sum[n]);
        }
    });
}
int eisen_hip_gemm_weight_gradients(eisen_ctx* ctx, size_t n, const void* const* A, const void* const* B, void* const* C, const size_t* M, const size_t* N, const int* accumulate,
                                    int dtype, size_t K) {
    const std::string before = ctx->order;
    for (size_t p = 0; p < n; p++) eisen_hip_gemm(ctx, A[p], B[p], C[p], dtype, EISEN_F32, 1, 0, M[p], N[p], K, accumulate[p]);
    ctx->order = before + 'w' + std::to_string(n);
    return 0;
}
int eisen_hip_gemm_residual(eisen_ctx* ctx, const void* A, const void* B, const void* R, void* C, int dtype_ab, int dtype_c, int ta, int tb, size_t M, size_t N, size_t K) {
    eisen_hip_dtod(ctx, C, R, M * N * (dtype_c == EISEN_BF16 ? 2 : 4));
    return eisen_hip_gemm(ctx, A, B, C, dtype_ab, dtype_c, ta, tb, M, N, K, 1);
}
// (h = gate * up: which function of them it is does not matter here)
int eisen_hip_swiglu(eisen_ctx* ctx, const void* gate, const void* up, void* h, int dtype, size_t n) {
    return give(ctx, [=] { for (size_t i = 0; i < n; i++) put(h, i, dtype, get(gate, i, dtype) * get(up, i, dtype)); });
}
int eisen_hip_gemm_swiglu_backward(eisen_ctx* ctx, const void* A, const void* B, const void* gate, const void* up, void* dgate, void* dup, int dtype, int ta, int tb, size_t M,
                                   size_t N, size_t K) {
    eisen_hip_gemm(ctx, A, B, dup, dtype, dtype, ta, tb, M, N, K, 0);
    return give(ctx, [=] {
        for (size_t i = 0; i < M * N; i++) {
            const float dh = get(dup, i, dtype);
            put(dgate, i, dtype, dh * get(up, i, dtype));
            put(dup, i, dtype, dh * get(gate, i, dtype));
        }
    });
}
int eisen_hip_gemm_weight_gradients_window(eisen_ctx* ctx, size_t n, size_t pieces, const void* const* A, const void* const* B, void* const* C, const size_t* M, const size_t* N, size_t K,
                                           const int* accumulate) {
    for (size_t p = 0; p < n; p++)
        for (size_t s = 0; s < pieces; s++)
            eisen_hip_gemm(ctx, A[p * pieces + s], B[p * pieces + s], C[p], EISEN_BF16, EISEN_F32, 1, 0, M[p], N[p], K, s > 0 || accumulate[p]);
    return 0;
}
int eisen_hip_gemm_forward_group(eisen_ctx* ctx, size_t n, const void* A, const void* const* B, void* const* C, const size_t* N, int dtype, size_t M, size_t K, size_t, size_t, size_t) {
    for (size_t p = 0; p < n; p++) eisen_hip_gemm(ctx, A, B[p], C[p], dtype, dtype, 0, 0, M, N[p], K, 0);
    return 0;
}
int eisen_hip_gemm_ksegments(eisen_ctx* ctx, size_t n, const void* const* A, const void* const* B, const size_t* K, void* C, int dtype_ab, int dtype_c, int ta, int tb, size_t M, size_t N,
                             int accumulate) {
    const std::string before = ctx->order;
    for (size_t p = 0; p < n; p++) eisen_hip_gemm(ctx, A[p], B[p], C, dtype_ab, dtype_c, ta, tb, M, N, K[p], p > 0 || accumulate);
    ctx->order = before + 's';
    return 0;
}
int eisen_hip_add(eisen_ctx* ctx, const void* a, const void* b, void* c, int dtype, size_t n) {
    return give(ctx, [=] { for (size_t i = 0; i < n; i++) put(c, i, dtype, get(a, i, dtype) + get(b, i, dtype)); });
}
int eisen_hip_accumulate(eisen_ctx* ctx, void* a, const void* b, int dtype, size_t n, int accumulate) {
    return give(ctx, [=] { for (size_t i = 0; i < n; i++) put(a, i, dtype, (accumulate ? get(a, i, dtype) : 0.f) + get(b, i, dtype)); });
}
// sections of side work, as runtime.hip has them
int eisen_hip_side_begin(eisen_ctx* ctx) {
    if (ctx->section) return -1;
    ctx->section = ctx->side = true;
    ctx->sides++;
    return 0;
}
int eisen_hip_side_begin_if_behind(eisen_ctx* ctx, int* forked) {
    if (ctx->section) return -1;
    ctx->section = true;
    *forked = ctx->side = *ctx->answers && *ctx->answers++ == '1';
    ++(*forked ? ctx->forks : ctx->inlines);
    return 0;
}
int eisen_hip_side_end(eisen_ctx* ctx) {
    if (!ctx->section) return -1;
    ctx->section = ctx->side = false;
    return 0;
}
int eisen_hip_side_wait(eisen_ctx* ctx) {
    if (ctx->section) return -1;
    for (auto& work : ctx->late) work();
    ctx->late.clear();
    return 0;
}
int eisen_hip_stream_sync(eisen_ctx* ctx) { return eisen_hip_side_wait(ctx); }
}

static std::vector<float> gradients(const char* answers, bool beside) {
    constexpr size_t kRows = 5, kHidden = 8;
    eisen_ctx ctx;
    ctx.answers = answers;
    std::vector<float> w(kHidden * kHidden), x(kRows * kHidden), seen;
    for (size_t i = 0; i < w.size(); i++) w[i] = (float)(i * 7 % 11) / 8 - 0.5f;
    for (size_t i = 0; i < x.size(); i++) x[i] = (float)(i * 5 % 13) / 4 - 1.5f;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Bf16Mixed);
    g.set_weight_gradients_beside(beside);
    const size_t wid = g.alloc({kHidden, kHidden}, w);
    g.mark_params();
    for (int pass = 0; pass < 2; pass++) {
        const size_t xid = g.alloc({kRows, kHidden}, x);
        g.backward(g.matmul(g.matmul(xid, wid), wid));
        for (size_t id : {wid, xid})
            for (size_t i = 0; i < g.at(id).size(); i++) seen.push_back(get(g.at(id).grad.ptr, i, g.at(id).grad.dtype));
        g.clear_activations();
    }
    if (beside && (ctx.forks + ctx.inlines != 4 || !ctx.late.empty())) throw eisen::Error("not the four sections that were meant");
    return seen;
}

static std::vector<float> ramp(size_t n, size_t step, size_t of, float scale) {
    std::vector<float> v(n);
    for (size_t i = 0; i < n; i++) v[i] = ((float)(i * step % of) - (float)(of / 2)) * scale;
    return v;
}

// Two weights, each used over few rows (left for the end of the pass) and W1 over many as well (beside the chain): P = S W2, Q = P W1, R = Q W2, Y = (X W1) R^T.
static std::vector<float> rows_of_two_lengths(const char* answers, bool beside) {
    constexpr size_t kFew = 8, kMany = 16392, kHidden = 32;
    eisen_ctx ctx;
    ctx.answers = answers;
    std::vector<float> seen;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Bf16Mixed);
    g.set_weight_gradients_beside(beside);
    const size_t w1 = g.alloc({kHidden, kHidden}, ramp(kHidden * kHidden, 7, 11, 0.125f)), w2 = g.alloc({kHidden, kHidden}, ramp(kHidden * kHidden, 5, 17, 0.0625f));
    g.mark_params();
    for (size_t w : {w1, w2}) g.request_zero_grad(w);
    const size_t s = g.alloc({kFew, kHidden}, ramp(kFew * kHidden, 5, 13, 0.25f)), x = g.alloc({kMany, kHidden}, ramp(kMany * kHidden, 3, 7, 0.5f));
    const size_t p = g.matmul(s, w2), many = g.matmul(x, w1), q = g.matmul(p, w1), r = g.matmul(q, w2);
    g.backward(g.matmul_trans_b(many, r));
    for (size_t id : {w1, w2, s})
        for (size_t i = 0; i < g.at(id).size(); i++) seen.push_back(get(g.at(id).grad.ptr, i, g.at(id).grad.dtype));
    g.clear_activations();
    if (beside && (ctx.forks + ctx.inlines == 0 || !ctx.late.empty())) throw eisen::Error("no section was meant to be left open, and one to be there");
    return seen;
}

// A weight large enough that the feed-forward tail forms its gradient on the side stream, used once more by the node behind it: R = X W, Y = R + (gate * up) W.
static std::vector<float> tail_and_its_residual(const char* answers, bool beside) {
    constexpr size_t kRows = 64, kIn = 256, kOut = 16384;
    eisen_ctx ctx;
    ctx.answers = answers;
    std::vector<float> seen;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Bf16Mixed);
    g.set_weight_gradients_beside(beside);
    const size_t w = g.alloc({kIn, kOut}, ramp(kIn * kOut, 7, 11, 0.125f));
    g.mark_params();
    g.request_zero_grad(w);
    std::vector<size_t> in;
    for (size_t i = 0; i < 3; i++) {
        in.push_back(g.alloc_pooled({kRows, kIn}));
        g.load_tensor_data(in.back(), ramp(kRows * kIn, 3 + 2 * i, 13, 0.25f).data(), kRows * kIn);
    }
    const size_t r = g.matmul(in[0], w), y = g.swiglu_matmul_residual(in[1], in[2], w, r);
    g.backward(y);
    if (ctx.sides == 0) throw eisen::Error("no work went to the side stream");
    // what both products add up to, whichever stream they ran on
    std::vector<float> got(kIn * kOut);
    for (size_t i = 0; i < got.size(); i++) got[i] = get(g.at(w).grad.ptr, i, EISEN_F32);
    for (size_t k = 0; k < kIn; k++) {
        float want = 0.f;
        for (size_t m = 0; m < kRows; m++)
            want += get(g.at(in[0]).data.ptr, m * kIn + k, EISEN_BF16) +
                    widen(narrow(get(g.at(in[1]).data.ptr, m * kIn + k, EISEN_BF16) * get(g.at(in[2]).data.ptr, m * kIn + k, EISEN_BF16)));
        for (size_t n = 0; n < kOut; n++)  // (dY is one everywhere, and every term a multiple of 1/16)
            if (got[k * kOut + n] != want) throw eisen::Error("the gradient is not the sum of both products");
    }
    seen = {1.f};
    g.clear_activations();
    return seen;
}

// A window of three passes over a layer that it holds and one too narrow for it, Y = (X W) V: what stays allocated behind a pass are the operands of W alone.
static std::vector<float> window_with_a_narrow_layer(const char* answers, bool beside) {
    constexpr size_t kRows = 128, kHidden = 1024, kNarrow = 32;
    eisen_ctx ctx;
    ctx.answers = answers;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Bf16Mixed);
    g.set_weight_gradients_beside(beside);
    const size_t w = g.alloc({kHidden, kHidden}, ramp(kHidden * kHidden, 7, 11, 0.125f)), v = g.alloc({kHidden, kNarrow}, ramp(kHidden * kNarrow, 5, 17, 0.0625f));
    g.mark_params();
    g.set_weight_gradient_window(3);
    for (size_t id : {w, v}) g.request_zero_grad(id);
    const size_t base = ctx.bytes();
    for (size_t pass = 1; pass <= 3; pass++) {
        const size_t x = g.alloc_pooled({kRows, kHidden});
        g.load_tensor_data(x, ramp(kRows * kHidden, 2 + pass, 13, 0.25f).data(), kRows * kHidden);
        g.backward(g.matmul(g.matmul(x, w), v));
        g.clear_activations();
        if (ctx.bytes() != base + (pass < 3 ? pass * 2 * kRows * kHidden * 2 : 0)) throw eisen::Error("pass " + std::to_string(pass) + ": not W's operands alone are kept");
    }
    std::vector<float> seen;
    for (size_t id : {w, v})
        for (size_t i = 0; i < g.at(id).size(); i++) seen.push_back(get(g.at(id).grad.ptr, i, EISEN_F32));
    return seen;
}

// When the products run: Y = ((X V) U) + ((X V) W), V alone, U and W as one node.  Kept to the tape, a node's products follow its input gradient and nothing is kept.
static std::vector<float> order_of_products(const char* answers, bool beside) {
    constexpr size_t kRows = 16, kHidden = 32;
    eisen_ctx ctx;
    ctx.answers = answers;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Bf16Mixed);
    g.set_weight_gradients_beside(beside);
    std::vector<size_t> w;
    for (size_t i = 0; i < 3; i++) w.push_back(g.alloc({kHidden, kHidden}, ramp(kHidden * kHidden, 3 + 2 * i, 11, 0.125f)));
    g.mark_params();
    const size_t x = g.alloc({kRows, kHidden}, ramp(kRows * kHidden, 3, 13, 0.25f));
    const size_t h = g.matmul(x, w[0]);
    const std::vector<size_t> both = g.matmul_group(h, {w[1], w[2]});
    const size_t y = g.add(both[0], both[1]);
    ctx.order.clear();
    g.backward(y);
    // (the group's input gradient is one call, s; V's product with X comes behind the input gradient of X)
    if (ctx.order != (beside ? "sdw3" : "sw2dw1")) throw eisen::Error("products ran in the order " + ctx.order);
    std::vector<float> seen;
    for (size_t id : w)
        for (size_t i = 0; i < g.at(id).size(); i++) seen.push_back(get(g.at(id).grad.ptr, i, EISEN_F32));
    return seen;
}

// Passes that throw when all their products are left: a gradient read behind one has them, one cleared behind one loses them, and the next pass is whole.  W is used over two
// numbers of rows: Y = (X W) ((S W) V)^T.
static std::vector<float> pass_that_threw(const char* answers, bool beside) {
    constexpr size_t kHidden = 32;
    eisen_ctx ctx;
    ctx.answers = answers;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Bf16Mixed);
    g.set_weight_gradients_beside(beside);
    const size_t w = g.alloc({kHidden, kHidden}, ramp(kHidden * kHidden, 7, 11, 0.125f)), v = g.alloc({kHidden, kHidden}, ramp(kHidden * kHidden, 5, 17, 0.0625f));
    g.mark_params();
    for (size_t id : {w, v}) g.request_zero_grad(id);
    const size_t base = ctx.bytes();
    std::vector<float> seen;
    auto read = [&](size_t id) {
        g.materialize_grad(id);
        for (size_t i = 0; i < g.at(id).size(); i++) seen.push_back(get(g.at(id).grad.ptr, i, EISEN_F32));
    };
    auto pass = [&](bool throws) {
        const size_t s = g.alloc({8, kHidden}, ramp(8 * kHidden, 5, 13, 0.25f)), x = g.alloc({16, kHidden}, ramp(16 * kHidden, 3, 7, 0.5f));
        if (throws) g.tape.nodes.push_back(eisen::TapeNode{{}, x, [](eisen::Graph&) { throw eisen::Error("meant"); }});
        const size_t y = g.matmul_trans_b(g.matmul(x, w), g.matmul(g.matmul(s, w), v));
        try {
            g.backward(y);
        } catch (const eisen::Error& e) {
            if (std::string(e.what()) != "meant") throw;
        }
    };
    pass(true);
    read(v);
    read(w);
    g.clear_activations();
    pass(true);
    for (size_t id : {w, v}) g.request_zero_grad(id);
    g.clear_activations();
    pass(false);
    read(w);
    read(v);
    g.clear_activations();
    pass(true);
    g.clear_activations();  // (nobody has asked for a gradient: the products are added before their operands go)
    read(v);
    read(w);
    if (ctx.bytes() != base) throw eisen::Error("operands are still allocated");
    return seen;
}

int main(int argc, char** argv) {
    if (argc < 2 || argc > 3) return 2;
    const char* answers = argv[argc - 1];
    const std::string graph = argc == 3 ? argv[1] : "weight_used_twice";
    try {
        const auto run = graph == "weight_used_twice" ? gradients : graph == "rows_of_two_lengths" ? rows_of_two_lengths : graph == "tail_and_its_residual" ? tail_and_its_residual
                         : graph == "window_with_a_narrow_layer" ? window_with_a_narrow_layer
                         : graph == "order_of_products" ? order_of_products
                         : graph == "pass_that_threw" ? pass_that_threw : nullptr;
        if (!run) return 2;
        const std::vector<float> plain = run("", false), beside = run(answers, true);
        bool some = false;
        for (float v : plain) some |= v != 0.f;
        if (!some || plain.size() != beside.size() || std::memcmp(plain.data(), beside.data(), plain.size() * sizeof(float))) {
            std::fprintf(stderr, "%s %s: gradients differ\n", graph.c_str(), answers);
            return 1;
        }
    } catch (const std::exception& e) {
        std::fprintf(stderr, "%s %s: %s\n", graph.c_str(), answers, e.what());
        return 1;
    }
    return 0;
}

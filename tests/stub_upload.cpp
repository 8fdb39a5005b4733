// Graph::load_tensor_data and Graph::gather on a stub of the device whose upload of values fails when it is told to: what a lookup is given afterwards.
// Exit status 0 if it is given the ids of the host's copy, all of them inside the vocabulary.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../eisen_amd/csrc/host/graph.hpp"

struct eisen_ctx {
    bool fails = false;
    std::vector<int32_t> looked_up;
};

extern "C" {
const char* eisen_hip_last_error(eisen_ctx*) { return "refused by the stub"; }
int eisen_hip_malloc(eisen_ctx*, size_t bytes, void** out) {
    if (!(*out = std::malloc(bytes + 16))) return -1;
    std::memset(*out, 0x7f, bytes);
    return 0;
}
int eisen_hip_malloc_zeroed(eisen_ctx*, size_t bytes, void** out) { return (*out = std::calloc(bytes + 16, 1)) ? 0 : -1; }
int eisen_hip_free(eisen_ctx*, void* p) { return std::free(p), 0; }
int eisen_hip_htod(eisen_ctx*, void* d, const void* s, size_t bytes) { return std::memcpy(d, s, bytes), 0; }
int eisen_hip_htod_values(eisen_ctx* ctx, void* d, int dtype, int32_t* ids, const float* s, size_t n) {
    if (ctx->fails || dtype != EISEN_F32) return -5;
    std::memcpy(d, s, n * sizeof(float));
    for (size_t i = 0; ids && i < n; i++) ids[i] = (int32_t)s[i];
    return 0;
}
int eisen_hip_gather(eisen_ctx* ctx, const void*, const int32_t* ids, void*, int, size_t n, size_t vocab, size_t) {
    ctx->looked_up.assign(ids, ids + n);
    for (size_t i = 0; i < n; i++)
        if (ids[i] < 0 || (size_t)ids[i] >= vocab) return -9;  // (the kernel would read past the weights)
    return 0;
}
int eisen_hip_side_wait(eisen_ctx*) { return 0; }
int eisen_hip_stream_sync(eisen_ctx*) { return 0; }
}

int main() {
    eisen_ctx ctx;
    eisen::Graph g(&ctx, eisen::PrecisionMode::Fp32);
    g.no_grad = true;
    const size_t w = g.alloc({3, 2}, std::vector<float>(6, 1.f));
    const std::vector<float> before = {90.f, 91.f, 92.f}, ids = {1.f, 0.f, 2.f};
    for (const bool loaded_before : {false, true}) {
        const size_t x = g.alloc_pooled({3});
        if (loaded_before) g.load_tensor_data(x, before.data(), 3);
        bool threw = false;
        ctx.fails = true;
        try {
            g.load_tensor_data(x, ids.data(), 3);
        } catch (const eisen::Error&) {
            threw = true;
        }
        ctx.fails = false;
        for (int turn = 0; turn < 2; turn++) {  // behind the load that failed, and behind one that did not
            try {
                g.gather(w, x);
            } catch (const eisen::Error& e) {
                std::fprintf(stderr, "loaded before %d, turn %d: %s\n", loaded_before, turn, e.what());
                return 1;
            }
            if (!threw || ctx.looked_up != std::vector<int32_t>{1, 0, 2}) {
                std::fprintf(stderr, "loaded before %d, turn %d: other ids were looked up\n", loaded_before, turn);
                return 1;
            }
            g.load_tensor_data(x, ids.data(), 3);
        }
    }
    return 0;
}

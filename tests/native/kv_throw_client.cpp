// A chunk of few rows under host memory that runs out: each of the library's own allocations in the call
// throws in turn. The call has to come back with a status, the layer has to count the rows it counted
// before, and the same call has to succeed afterwards. Exit status 0 = so it was.
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include <dlfcn.h>

#include "saragossa_kv.h"

static int armed = -1; // allocations of the library that still succeed; -1 = all

// (the runtime's and the standard library's own allocations pass)
static bool from_library(void *caller) {
    Dl_info info;
    return dladdr(caller, &info) && info.dli_fname && std::strstr(info.dli_fname, "libsaragossa_kv");
}
void *operator new(std::size_t n) {
    if (armed >= 0 && from_library(__builtin_return_address(0)) && armed-- == 0) throw std::bad_alloc();
    void *p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

#define CHECK(cond, what)                                                                             \
    do {                                                                                              \
        if (!(cond)) {                                                                                \
            std::fprintf(stderr, "FAIL %s (line %d): %s\n", what, __LINE__, skv_last_error());        \
            return 1;                                                                                 \
        }                                                                                             \
    } while (0)

int main() {
    const size_t q_heads = 32, kv_heads = 8, head_dim = 64, base = 600, rows = 6;
    const size_t kv_dim = kv_heads * head_dim, q_dim = q_heads * head_dim;
    std::vector<float> kv((base + rows) * kv_dim), q(rows * q_dim), out(rows * q_dim);
    for (size_t i = 0; i < kv.size(); ++i) kv[i] = (float)((i * 2654435761u >> 9) % 1000) / 500.0f - 1.0f;
    for (size_t i = 0; i < q.size(); ++i) q[i] = kv[(i * 7 + 3) % kv.size()];
    skv_ctx *ctx = nullptr;
    skv_layer *layer = nullptr;
    CHECK(skv_ctx_create(0, &ctx) == SKV_OK, "ctx_create");
    CHECK(skv_layer_create(ctx, base + rows, q_heads, kv_heads, head_dim, SKV_DTYPE_BF16, 0, &layer) == SKV_OK, "layer_create");
    CHECK(skv_seed(layer, kv.data(), kv.data(), base * kv_dim, base) == SKV_OK, "seed");
    const float *fresh = kv.data() + base * kv_dim;
    int failed = 0;
    for (;; ++failed) {
        CHECK(failed < 16, "the call allocates without end");
        armed = failed;
        const int32_t rc = skv_prefill_chunk_host(layer, q.data(), fresh, fresh, rows, out.data());
        const bool threw = armed < 0;
        armed = -1;
        if (!threw) {
            CHECK(rc == SKV_OK, "chunk");
            break;
        }
        CHECK(rc == SKV_ERR_DEVICE, "chunk without memory");
        CHECK(skv_len(layer) == base, "rows counted that nobody wrote");
    }
    CHECK(failed > 0, "no allocation was made to fail");
    CHECK(skv_len(layer) == base + rows, "len");
    std::printf("%d allocations failed\nok\n", failed);
    skv_layer_destroy(layer);
    skv_ctx_destroy(ctx);
    return 0;
}

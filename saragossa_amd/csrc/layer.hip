// Host side of one layer's paged KV cache: the stand-in for FullAttentionMetalState
// (src/decode_resident/attention.rs:457-1038). All bookkeeping (len, block table)
// lives on the host and advances at call time, before the GPU has run the work,
// exactly like the reference's encode-time `len += 1` (attention.rs:993).
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <new>
#include <string>
#include <vector>

#include "layer.h"

namespace skv {

static thread_local std::string g_last_error;

void set_error(const std::string &msg) { g_last_error = msg; }
int32_t fail(int32_t code, const std::string &msg) {
    g_last_error = msg;
    return code;
}
int32_t fail_hip(hipError_t e, const char *what) {
    g_last_error = std::string("HIP: ") + hipGetErrorString(e) + " (" + what + ")";
    return SKV_ERR_DEVICE;
}

hipError_t arena_get(skv_ctx *ctx, size_t bytes, void **ptr, size_t *got) {
    *ptr = nullptr;
    *got = 0;
    if (bytes == 0) bytes = 256;
    {
        std::lock_guard<std::mutex> lk(ctx->arena_mu);
        auto it = ctx->arena_free.lower_bound(bytes);
        if (it != ctx->arena_free.end() && it->first <= bytes + bytes / 4) {
            *ptr = it->second;
            *got = it->first;
            ctx->arena_bytes -= it->first;
            ctx->arena_free.erase(it);
            return hipSuccess;
        }
    }
    const hipError_t e = hipMalloc(ptr, bytes);
    if (e == hipSuccess) *got = bytes;
    return e;
}

void arena_put(skv_ctx *ctx, void *ptr, size_t bytes) {
    if (!ptr) return;
    ctx->scratch.freed(); // (or about to be, in a layer's end: worth another question at most)
    {
        std::lock_guard<std::mutex> lk(ctx->arena_mu);
        if (!ctx->closed && ctx->arena_bytes + bytes <= ctx->arena_cap) {
            ctx->arena_free.emplace(bytes, ptr);
            ctx->arena_bytes += bytes;
            return;
        }
    }
    (void)hipFree(ptr);
}

// The device as a context's scratch sees it. A failed call leaves no error behind for the next launch to report.
static struct HipScratch final : ScratchDevice {
    static int status(hipError_t e) {
        if (e != hipSuccess) (void)hipGetLastError();
        return (int)e;
    }
    int alloc(void **p, size_t bytes) override { return status(hipMalloc(p, bytes)); }
    int free(void *p) override { return status(hipFree(p)); }
    int wait_stream(void *stream) override { return status(hipStreamSynchronize(static_cast<hipStream_t>(stream))); }
    int wait_device() override { return status(hipDeviceSynchronize()); }
    bool full(int status) override { return status == (int)hipErrorOutOfMemory; }
} hip_scratch;

// Frees what the context holds on the device; the caller has synchronised the device.
static void ctx_drain(skv_ctx *ctx) {
    ctx->scratch.drain(hip_scratch);
    std::lock_guard<std::mutex> lk(ctx->arena_mu);
    for (auto &kv : ctx->arena_free) (void)hipFree(kv.second);
    ctx->arena_free.clear();
    ctx->arena_bytes = 0;
}

void ctx_release(skv_ctx *ctx) {
    if (ctx->refs.fetch_sub(1, std::memory_order_acq_rel) != 1) return;
    // a layer that outlived skv_ctx_destroy may have grown the multi-query scratch again
    if (!ctx->scratch.empty()) {
        (void)hipSetDevice(ctx->device);
        (void)hipDeviceSynchronize();
        ctx_drain(ctx);
    }
    delete ctx;
}

} // namespace skv

using namespace skv;

// Split-K partials of skv_decode_step_static_device, for callers that cannot allocate. Every
// GPU the library runs on holds its own copy of the array until the process ends. In host
// code the array's name is only a stand-in: its device address comes from
// hipGetSymbolAddress, once per device (static_scratch_ptr), and only that pointer is ever
// handed to a kernel.
static __device__ __align__(256) unsigned char scratch[SKV_STATIC_SCRATCH_BYTES];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[MAX_DEVICES] = {};

// The device address of `scratch` on `device`, which must be the current device.
hipError_t static_scratch_ptr(int device, void **ptr) {
    *ptr = nullptr;
    if (device < 0 || device >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[device] = p;
    }
    *ptr = g_scratch_ptr[device];
    return hipSuccess;
}

// Dims of a tile's row: whole K-steps of 32, where kernels are built for them. (96 for the heads of 65 to 96 dims: with 128, a
// quarter of their bytes and products was padding.)
int padded_head_dim(size_t hd) {
    for (int p : {32, 64, 96, 128, 256, 512})
        if ((size_t)p >= hd) return p;
    return 0;
}
// Elements of a row that a layer's pools have room for: a power of two, as callers who budget by skv_layer_bytes know it.
size_t pool_head_dim(size_t hd) {
    size_t p = 32;
    while (p < hd) p *= 2;
    return p;
}

size_t env_usize(const char *name, size_t dflt) {
    const char *raw = std::getenv(name);
    if (!raw || !*raw) return dflt;
    char *end = nullptr;
    unsigned long long v = std::strtoull(raw, &end, 10);
    if (end == raw) return dflt;
    return (size_t)v;
}

// Launch-shaping knobs from the environment, read once per flag generation
// (skv_flags_reload starts a new one), not once per launch.
struct Tuning {
    size_t split_min_len;   // rows below which the context is not split
    bool split_min_len_given;
    size_t target_wgs;      // workgroups a decode launch aims for
    bool wgs_given;         // that or prefill_wgs
    size_t min_pages;       // pages per split at least (0 = one per wavefront)
    size_t forced_waves;    // 4 or 8, 0 = by shape
    bool q_vec, fused_append;
    size_t prefill_tiles;   // 0 = never, 1 = by shape, 2 = every chunk of 64 query slots and more
    size_t prefill_wgs, prefill_max_splits;
    long prefill_tiles2_min_pages; // -1 = by head_dim
    size_t f32_terms;       // f32 chunks: 0 = every workgroup splits its pages into terms, 1 = by shape, 2 = a launch of its own does
    size_t f32_terms_max;   // bytes of terms that a context holds
};

const Tuning &tuning() {
    thread_local Tuning t{};
    thread_local uint64_t seen = 0;
    const uint64_t epoch = skv_internal_flags_epoch();
    if (epoch != seen) {
        t.split_min_len = skv_effective_split_min_len();
        t.split_min_len_given = std::getenv("RETI_RUST_SDPA_2PASS_MIN_LEN") != nullptr;
        t.target_wgs = std::max<size_t>(env_usize("SKV_DECODE_WGS", 256), 1);
        t.wgs_given = std::getenv("SKV_DECODE_WGS") != nullptr || std::getenv("SKV_PREFILL_WGS") != nullptr;
        t.min_pages = env_usize("SKV_DECODE_MIN_PAGES", 0);
        t.forced_waves = env_usize("SKV_DECODE_WAVES", 0);
        t.q_vec = env_usize("SKV_Q_VEC", 1) != 0;
        t.fused_append = env_usize("SKV_FUSED_APPEND", 1) != 0;
        t.prefill_tiles = env_usize("SKV_PREFILL_TILES", 1);
        t.prefill_wgs = std::max<size_t>(env_usize("SKV_PREFILL_WGS", 256), 1);
        t.prefill_max_splits = std::max<size_t>(env_usize("SKV_PREFILL_MAX_SPLITS", 512), 1);
        t.prefill_tiles2_min_pages = std::getenv("SKV_PREFILL_TILES2_MIN_PAGES")
                                         ? (long)env_usize("SKV_PREFILL_TILES2_MIN_PAGES", 0) : -1;
        t.f32_terms = env_usize("SKV_F32_TERMS", 1);
        t.f32_terms_max = std::min<size_t>(env_usize("SKV_F32_TERMS_MB", 512), 1 << 20) << 20;
        seen = epoch;
    }
    return t;
}

// Wavefronts per workgroup of the split kernel. Eight halve the number of partials for the
// same number of wavefronts in flight; four are better when eight would leave three
// quarters of the compute units without a workgroup (short contexts, ring layers).
int choose_waves(const skv_layer *L, int n_pages_scan) {
    if (L->g.P > 256) return 4; // one wavefront per SIMD: 512 registers each
    const size_t forced = tuning().forced_waves;
    if (forced == 4 || forced == 8) return (int)forced;
    const size_t kvh = (size_t)L->g.kv_heads;
    const size_t wgs8 = kvh * std::max<size_t>(std::min<size_t>(256 / std::max<size_t>(kvh, 1), (size_t)n_pages_scan / 8), 1);
    return wgs8 <= 64 && n_pages_scan >= 8 ? 4 : 8;
}

size_t decode_target_wgs() { return tuning().target_wgs; }

// Shape of the prefill tile kernel's workgroups for a chunk of n_slots query slots per kv head, each
// walking about n_pages pages. Workgroups of halves or quarters cover 64 slots instead of 128, so they fill
// the device with fewer splits, or with none where 128-slot workgroups need two and a merge; they
// copy each page for half as many slots. Quarters (head_dim 65 to 128) read LDS half as often per product as
// halves but walk eight pages at a time and join four states. Two tiles read LDS half as often too, and need
// the most splits: they pay on long walks. Above 256 workgroups of 64 slots the device is full in any shape. The lines are in pages walked
// by all 64-slot workgroups, where whole chunks cost the same in two shapes, between layers that are not in any cache and those that are, as a
// short prompt's, where halves stay ahead for longer (512 rows of q32/kv8/hd64 over 2000, halves / two tiles 29.5/36.1 in
// caches, 34.8/36.2 not; of q32/kv8/hd128 over 1024, halves / quarters 34.5/34.9 and 34.4/36.3, over 2048 46.8/47.6 and 50.5/46.8). On layers
// in no cache, over 181 chunks of 64 to 1024 rows with up to 256 workgroups, the shape chosen is 1.7 % slower than the best on the average, at most 14 %
// (400 to 600 rows of hd128 heads at walks of 20000 to 29000, where halves are up to 13 % behind quarters; in caches the two are even). Above 256
// workgroups, over 33 chunks, 10 % and 42 %: the line of two tiles stands too high for 257 to 350 of them (700 rows of q28/kv4/hd128 over
// 4000, 8000, one tile / two 119/92, 210/149). One tile / two tiles / halves / quarters, in us on one MI355X, in no cache, with workgroups, walk in thousands: q32/kv8/hd128, 400 rows over 500, 1500, 3000, 6000 (200; 11, 24, 43,
// 80) 32.5/37.2/25.0/27.2, 42.7/44.5/40.0/37.6, 59.5/59.7/64.0/55.0, 94.4/90.2/110/87.9, 512 over 1500, 6000 (256; 32, 104)
// 48.0/49.8/42.8/40.8, 106/100/114/96.2; q28/kv4/hd128, 400 over 500, 1500, 6000 (176; 10, 21, 70) 31.8/36.6/23.8/26.3, 42.6/43.2/38.6/36.4,
// 92.2/79.1/107/85.1; q24/kv8/hd128, 400 over 1500, 3000, 6000 (152; 18, 32, 61) 35.7/41.2/39.6/37.0, 48.5/51.5/63.4/54.3, 74.8/74.5/109/87.2, 512
// over 3000, 6000 (192; 42, 78) 60.7/58.6/65.3/56.4, 94.9/84.8/112/89.1, 1024 over 1500 (384) 71.6/77.6/75.8/76.9; q32/kv8/hd64, 400 over 1500, 3000,
// 6000 (200; 24, 43, 80) 29.8/31.7/28.2, 40.7/40.5/45.0, 63.2/57.8/75.8, 256 over 3000, 12000 (128; 26, 98) 29.1/32.5/30.5, 63.0/61.5/79.0;
// q16/kv2/hd256 (one tile / halves), 400 over 3000, 6000 (100; 21, 40) 60.8/59.9, 87.5/92.4, 1024 over 1500, 6000 (256; 40, 112) 85.9/73.7, 191/186.
// (Two tiles fill the device in five splits up to 204 workgroups; from there to 256 only four fit, and up to 48 compute units stay idle:
// quarters stay ahead of them for longer there.) Heads of 65 to 96 dims walk a pair in less time, so that joining the states weighs more and the
// reads of LDS less. q12/kv4/hd96, 512 rows over 4096, 16000 (96; 28, 98) 36.5/40.9/45.2/41.0, 82.7/80.4/129/101, 1024 rows over 300, 1000, 2048, 4096
// (192; 16, 24, 37, 61) 31.6/35.5/25.1/26.8, 37.5/39.8/34.7/33.2, 46.5/45.9/48.3/42.9, 64.9/58.6/75.5/62.1; q30/kv10/hd96, 448 over 500, 1200, 3000, 5000
// (210; 13, 22, 45, 72) 27.7/33.0/22.8/24.7, 33.8/37.2/32.3/31.1, 51.0/51.8/56.9/48.7, 69.8/68.9/85.7/68.8.
TileShape prefill_shape(const Geom &g, size_t n_slots, size_t n_pages) {
    if (g.P > 256) return TileShape::one_tile;
    const long knob = tuning().prefill_tiles2_min_pages;
    if (knob >= 0) return g.P <= 128 && (long)n_pages >= knob ? TileShape::two_tiles : TileShape::one_tile;
    const size_t wgs = (n_slots + 63) / 64 * (size_t)g.kv_heads, walk = wgs * n_pages;
    if (wgs > 256) return g.P <= 128 && walk >= 250000 ? TileShape::two_tiles : TileShape::one_tile;
    if (g.P <= 64) {
        if (walk < (wgs >= 192 ? 46000u : 26500u)) return TileShape::halves;
        return wgs >= 192 || walk >= 90000 ? TileShape::two_tiles : TileShape::one_tile;
    }
    if (g.P > 128) return walk < (wgs >= 192 ? 130000u : 40000u) ? TileShape::halves : TileShape::one_tile;
    const bool p96 = g.P <= 96;
    if (wgs < (p96 ? 192u : 172u)) return walk < (p96 ? 20000u : 16000u) ? TileShape::halves : walk < 70000 ? TileShape::one_tile : TileShape::two_tiles;
    if (walk < (p96 ? 24000u : wgs >= 208 ? 30000u : 19000u)) return TileShape::halves;
    const size_t quarters_to = p96 ? (wgs >= 208 ? 75000 : 50000) : wgs >= 208 ? 105000 : wgs >= 196 ? 85000 : 55000;
    return walk < quarters_to ? TileShape::quarters : TileShape::two_tiles;
}

// Whether a chunk of n_queries rows over n_pages pages takes the kernel that shares each page among 64 to 256 query slots
// through LDS, or the decode kernel's multi-query mode (speculative verify rows, short chunks over short contexts): one workgroup
// per 16 slots that streams the pages into its own registers, without a prologue to speak of, but asks for every page once per 16
// slots. The line is the number of (16 slots, page) pairs, as a chunk's rows walk them on the average, where those requests cost
// what the tile kernel's start does. It depends on how the workgroups of either fall on the 256 compute units:
// - the multi-query mode's, one to a compute unit: it loses early where two splits and their merge have to make up for few tiles (86 to 128 of
//   16 slots), or where the last round of workgroups leaves more than a third of the device idle;
// - the tile kernel's 64-slot ones: from 129 on they need no split and no merge, from 193 to 256 they fill the device in one round; above, they
//   are of 128 slots.
// Over 1955 chunks of 12 to 1024 rows around the lines in nineteen geometries, on layers in no cache, the kernel chosen is 0.6 % slower than the
// better one on the average (P 512: 1 %), 15 % at most. Multi-query mode / tile kernel, in us on one MI355X, with the pairs they walk in thousands:
// q32/kv8/hd128, no such trouble: 128 rows (256 tiles) 30 20.9/24.6, 54 30.9/30.5; two splits: 64 rows (128) 18 22/23.0, 30 28/26.5; a third idle:
// 160 rows (320) 18 21.7/22.4, 30 28.4/25.6; unsplit tiles: 384 rows (192 workgroups of 64) 18 18.5/18.4, 37 25.8/24.4; one round:
// 512 rows (256) 16 19.5/17.0, 37 27.9/22.7, q28/kv4/hd128, 448 rows (196) 12 18.0/16.5, 37 30.7/24.2; above: 600 rows (304) 31
// 26.9/27.8, 44 33.1/32.3. q16/kv2/hd256, 256 rows (256 tiles) 18 23.6/30.2, 33 33.8/35.5; 128 rows (128) 9 27.6/26.7, 23 36.7/32.4; 320 rows
// (320) 14 28.7/28.7, 23 37.1/31.6; 700 rows (176 workgroups) 16 31.0/27.3, 33 44.4/35.7. q8/kv2/hd512, 32 rows (16 tiles) 4.5 37.2/46.0; 128 rows
// (64) 3.7 38.9/41.0, 5.6 46.8/41.7; 200 rows (100, two splits) 1.3 37.7/33.3; 320 rows (160) 3.2 36.8/42.2, 5.6 49.0/44.4; 600 (300) 6 56.8/44.9.
// (With one line per size of head, 448 rows of q28/kv4/hd128 over 516 took 30.8, 100 rows of q16/kv8/hd256 over 4108 48.0, 32 of q8/kv2/hd512 over
// 4500 46.1: now 24.2, 37.1, 36.9.)
bool takes_tile_kernel(const Geom &g, size_t n_queries, size_t n_pages) {
    const size_t n_slots = n_queries * (size_t)g.gqa;
    if (tuning().prefill_tiles != 1 || n_slots < 64) return tuning().prefill_tiles > 1 && n_slots >= 64;
    const size_t wgs = (n_slots + 63) / 64 * (size_t)g.kv_heads, tiles = (n_slots + 15) / 16 * (size_t)g.kv_heads;
    const size_t walked = n_pages > n_queries / 32 ? n_pages - n_queries / 32 : 1, pairs = tiles * walked;
    if (g.P > 256) return pairs >= (tiles <= 36 ? 6000u : tiles <= 85 ? 4200u : tiles <= 128 ? 1100u : tiles <= 256 ? 5200u : 3000u);
    struct Lines {
        size_t full, two_splits, third_idle, unsplit, one_round, many;
    };
    const Lines l = g.P <= 32    ? Lines{44000, 35500, 29500, 15500, 12000, 32000}
                    : g.P <= 64  ? Lines{51500, 34300, 34300, 17300, 12000, 34500}
                    : g.P <= 96  ? Lines{50000, 25500, 31500, 25500, 12000, 33000}
                    : g.P <= 128 ? Lines{44000, 30000, 26500, 18500, 12000, 37500}
                                 : Lines{26000, 9000, 13700, 9000, 9000, 20000};
    if (wgs > 256) return pairs >= l.many;
    if (wgs > 192) return pairs >= l.one_round;
    if (wgs > 128) return pairs >= l.unsplit;
    if (tiles <= 128) return pairs >= (tiles > 85 ? l.two_splits : l.full);
    return pairs >= (3 * tiles < 2 * 256 * ((tiles + 255) / 256) ? l.third_idle : l.full);
}

// The same questions for f32 layers: the kernel that splits its factors into bf16 terms (head_dim up to
// 256) or the one that streams pages into the f32 instruction, 16 slots a workgroup. The line is in (16 slots,
// page) pairs as a chunk's rows walk them on the average, each up to its own position: half of the pages of a
// first chunk (counted by all pages, 384 rows of q16/kv2/hd256 over 100 took the first kernel, 82.5 us, where
// streaming takes 52.2, and 512 over none 58.8 where it takes 51.1), lower where 64-slot workgroups fill the device without a split.
// Over 937 chunks of 64 to 1024 rows around the lines in ten geometries the kernel chosen is 1 % slower than the other on the average, at most 27 % (384
// rows of q32/kv8/hd128 over 52, 192 workgroups of 64 slots). Whole chunks,
// streaming / the kernel of terms, in us, with the pairs they walk in thousands: q32/kv8/hd128, 512 rows over none (16; 256 workgroups)
// 40.4/31.1, 416 (11; 208) 34.2/27.8, 64 over 1000, 2000 (8, 16) 25.7/30.7, 36.0/34.1, 128 over 300, 1000 (6, 17) 23.4/32.3, 37.5/33.4, 256 over
// 300 (14) 31.3/34.5; q24/kv8/hd128, 128 over 1000 (13) 36.7/31.9; q12/kv4/hd96, 256 over 1000 (14) 30.7/26.9, 128 over 2000 (12) 27.6/28.5;
// q8/kv8/hd80, 64 over 8000 (16) 36.1/40.3; q8/kv2/hd64, 256 over 2000, 4000 (17, 33) 22.0/24.7, 32.6/30.8, 512 over 300, 1000 (9, 20)
// 18.1/20.9, 25.1/22.9; q32/kv8/hd64, 416 over none (11; 208) 19.8/18.6, 160 over 1000 (22) 30.7/26.1; q16/kv2/hd256, 128 over 1000, 2000
// (9, 17) 50.7/61.5, 71.7/64.0; q32/kv8/hd32, 512 over none (16; 256) 14.7/15.7; where streaming fills its round, or is of few tiles, q32/kv8/hd128, 256
// over 312 (14; 512 tiles) 31.8/34.2, 160 over 600 (14; 320) 38.6/30.9, q32/kv8/hd64, 350 over 312 (23; 704) 26.1/28.0, q8/kv2/hd64, 64 over
// 11800 (24; 64) 32.3/34.2.
bool takes_f32_chunk_kernel(const Geom &g, size_t n_queries, size_t n_pages) {
    const size_t n_slots = n_queries * (size_t)g.gqa;
    if (f32_prefill_slots(g.P, false) == 0 || n_slots < 64 || tuning().prefill_tiles == 0) return false;
    if (tuning().prefill_tiles > 1) return true;
    const size_t wgs = (n_slots + 63) / 64 * (size_t)g.kv_heads;
    const size_t tiles = (n_slots + 15) / 16 * (size_t)g.kv_heads;
    // (512 tiles of 16 slots are one full round of streaming workgroups, two to a compute unit)
    size_t line = g.P <= 32    ? 26000
                  : g.P <= 64  ? (tiles <= 85 || tiles > 384 ? 25000 : 21500)
                  : g.P <= 96  ? 16200
                  : g.P <= 128 ? (tiles > 448 && tiles <= 512 ? 15000 : 12600)
                               : 12200;
    if (g.P > 32 && wgs >= 208 && wgs <= 256) line = std::min<size_t>(line, 10000);
    const size_t walked = n_pages > n_queries / 32 ? n_pages - n_queries / 32 : 1;
    return tiles * walked >= line;
}
bool f32_halves(const Geom &g, size_t n_slots, size_t n_pages) {
    if (tuning().prefill_tiles2_min_pages >= 0) return false;
    const size_t wgs = (n_slots + 63) / 64 * (size_t)g.kv_heads, walk = wgs * n_pages;
    if (n_slots <= 64) return true; // a workgroup of 128 slots would be half empty
    return wgs <= 256 && walk < (g.P <= 64 ? 17000u : wgs >= 192 ? 25000u : 8500u);
}

// Splits of the context for a chunk whose workgroups cover per_wg slots: while the slot tiles alone
// leave compute units idle, and at least 16 pages each.
int chunk_splits(const Geom &g, size_t n_queries, size_t per_wg, size_t n_pages) {
    if (!skv_flag_sdpa_2pass_enabled()) return 1;
    const size_t tiles = (n_queries * (size_t)g.gqa + per_wg - 1) / per_wg * (size_t)g.kv_heads;
    size_t want = std::max<size_t>(tuning().prefill_wgs / tiles, 1);
    want = std::min<size_t>(want, std::max<size_t>(n_pages / 16, 1));
    return (int)std::min<size_t>(want, tuning().prefill_max_splits);
}

// Splits of a launch in which the workgroups of several query tiles walk the same pages. Workgroup ids, the split fastest,
// then the kv head, go to the eight XCDs in turn: where splits x kv heads are whole eights, all tiles of a
// (split, kv head) run on one XCD and its L2 has a page from memory once. Worth up to a tenth of the splits: rows of
// q16/kv2/hd256 as whole chunks on layers in no cache, in us, splits as they are / in whole eights, 6 over 8192 (42/40)
// 15.6/14.7, over 20000 22.5/19.9, 12 over 8192 (21/20) 21.0/17.1; with plain loads 18 over 4000 (14/12) 16.9/17.6, 23 (11/8)
// 17.5/17.8, 36 (7/4) 20.5/22.7. On f32 layers (42/40 and 21/20) 6 over 20000 88.5/80.4, 12 over 8192 61.6/58.5, but 24 of q28/kv4/hd128
// (11/10) over 1356, 3420 23.6/24.3, 32.0/33.1, 28 of q24/kv4/hd256 over 1356 1/1.10: there a sixteenth (`share`).
// Not where the wavefronts of a workgroup are four (f32 layers, heads above 256 dims), have a page each and would walk a second one: 12
// rows of q8/kv2/hd512 over 1300 (21/20 splits of 83 pages) 20.9/22.8, on f32 layers 35.7/42.9, 30 of q16/kv2/hd256 over 1042
// (17/16 of 67) on f32 34.1/36.5. (Where they walk two already fewer splits gain: 12 rows of q8/kv2/hd512 on f32 over 2680 65.2/52.5; and
// eight wavefronts gain in any case, 6 rows of q16/kv2/hd256 over 2630, 42/40 of 165, 13.6/12.9.)
int xcd_splits(int splits, int kv_heads, int n_pages, int waves, int share) {
    int unit = 8;
    for (int h = kv_heads; unit > 1 && h % 2 == 0; h /= 2) unit /= 2;
    const int fewer = splits - splits % unit;
    if (splits % unit * share > splits || (waves == 4 && n_pages <= splits * 4 && n_pages > fewer * 4)) return splits;
    return fewer;
}

int choose_splits(const skv_layer *L, int n_pages_scan, size_t rows, int waves, size_t target_wgs) {
    const Tuning &t = tuning();
    if (!skv_flag_sdpa_2pass_enabled() || rows < t.split_min_len) return 1;
    const size_t min_pages = std::max<size_t>(t.min_pages ? t.min_pages : (size_t)waves, 1);
    size_t s = std::max<size_t>(target_wgs / (size_t)L->g.kv_heads, 1);
    // Short contexts: as many splits as leave no split more than min_pages pages (rounded up,
    // not down: with one page per wavefront no wavefront then walks a second page, which
    // would be a whole memory latency more for the launch).
    s = std::min<size_t>(s, ((size_t)n_pages_scan + min_pages - 1) / min_pages);
    s = std::min<size_t>(s, (size_t)L->max_splits);
    return (int)std::max<size_t>(s, 1);
}

// Contexts of so few pages that one workgroup to a tile of query slots, with no split, is done before the merge of a split would be:
// a launch less for the host too. Not where a knob of the splits is set, nor where the context lies over what the launch reads.
bool may_stay_whole() {
    const Tuning &t = tuning();
    return !t.split_min_len_given && !t.wgs_given && t.min_pages == 0 && t.forced_waves == 0;
}
bool overlap(const void *a, size_t a_bytes, const void *b, size_t b_bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + b_bytes && y < x + a_bytes;
}
// Whether the context of n rows lies over queries that workgroups other than the one that writes it may still have to read. An unsplit
// launch, whose first workgroups write while others have yet to start, then writes elsewhere (see encode_attention); a split one's merge
// starts behind all reads. Exactly in the queries' place it may lie: a workgroup reads the rows of its own slots alone, and writes
// them when it has (but for one kernel, see reads_again). head_stride: elements between the heads of the queries (0 = head_dim).
bool over_queries(const Geom &g, const float *out, const float *q, size_t n, size_t head_stride = 0) {
    const size_t bytes = n * (size_t)g.q_heads * g.head_dim * sizeof(float);
    if (out == q && head_stride == 0) return false;
    return overlap(out, bytes, q, head_stride ? (size_t)g.q_heads * head_stride * sizeof(float) : bytes);
}
// The f32 chunk kernel on heads above 128 dims: its plain_slot comes back to a query row after half of the context's columns are stored.
bool reads_again(const Geom &g, const float *out, const float *q) { return g.f32 && g.P > 128 && out == q; }
// The same for n K or V rows.
bool over_rows(const Geom &g, const float *out, const float *rows, size_t n) {
    return rows && overlap(out, n * (size_t)g.q_heads * g.head_dim * sizeof(float), rows, n * (size_t)g.kv_heads * g.head_dim * sizeof(float));
}
// Decode steps of bf16 layers, eight wavefronts a workgroup. Split / whole, us of GPU time on one MI355X: q32/kv8/hd128 over 150, 250, 380 rows
// 6.5/5.2, 6.4/5.6, 6.4/6.8; q8/kv8/hd80 6.3/4.9, 6.2/5.0, 6.3/5.9, 500 6.3/6.7; q8/kv2/hd64 5.7/4.5, 5.7/4.6, 5.8/5.2, 500 5.8/5.7; q16/kv2/hd256 7.8/7.1,
// 7.8/8.1; with the pre-KV step q16/kv8/hd256 over 150 9.6/8.7. Calls in a stream, where the host's two launches take longer than the
// device: q32/kv8/hd128 over 250 9.1/7.1. (f32 layers, q32/kv8/hd128 over 140, 250 7.6/7.7, 7.6/9.8.)
// In a batch whose contexts all stay whole the line rises with its workgroups (batch_wgs, sequences times kv heads; 0 = no batch): the more there are,
// the fewer splits would share the device. Batches, split / whole: q8/kv8/hd80, 4 over 380, 500 rows 7.1/6.3, 7.1/7.3, 8 over 500, 700 8.0/7.6,
// 8.8/9.0, 16 over 500, 700, 1500 10.0/8.2, 11.6/9.7, 16.5/16.5; q32/kv8/hd128, 4 over 380, 500 7.6/7.3, 7.8/8.5, 8 over 380, 500 9.0/7.7, 9.3/8.9,
// 16 over 500, 700 12.0/9.7, 14.8/12.1; q16/kv4/hd128, 16 over 500, 700 9.4/9.0, 10.6/10.7; q8/kv8/hd128, 3 over 350 7.0/7.2, 8 over 510 8.7/8.9; q16/kv8/hd256, 4 over
// 150, 250 8.6/7.5, 8.5/9.0, 8 over 250, 380 10.2/9.4, 11.8/11.5, 16 over 250, 380 12.8/10.7, 15.7/13.5. (f32, q32/kv8/hd128: 8 over 250
// 10.0/10.6, 16 over 380 16.3/15.1, 16 over 3000 69.8/71.6.)
// The line in pages, 0 = none stays whole.
int whole_step_pages(const Geom &g, int batch_wgs) {
    if (!may_stay_whole() || g.f32 || g.P > 256) return 0;
    return g.P <= 96 ? 24 + batch_wgs / 5 : g.P <= 128 ? 16 + batch_wgs / 5 : 10 + std::max(batch_wgs - 32, 0) / 6;
}
// Chunks in the multi-query mode, of `tiles` tiles of all kv heads: the more there are, the fewer splits would share the device. Split / whole, us of GPU
// time: q32/kv8/hd128, 6 rows (16 tiles) over 250, 490 8.5/6.3, 8.5/8.1, 30 (64) over 250, 700, 900 12.2/8.1, 12.9/11.4, 12.6/12.1, 60 (120) over 1300
// 17.0/15.2; q8/kv2/hd64, 6 (4) over 440 6.9/6.2, 60 (30) over 600 8.8/7.6; q16/kv2/hd256, 48 (48) over 460 14.9/12.7, 90 (90) over 650 20.0/15.1.
// Tiles of a kv head walk the same pages, on one or two XCDs where kv heads are whole fours (`near`), else on four or eight. Whole, every one of those then asks
// memory for each page, unless the launch loads shared pages (pages_shared: more than four tiles, never where it appends the rows). There, and where a tile walks
// alone, the line is lower: q24/kv1/hd128, 6 rows (9 tiles) over 330, 380, 470 8.8/8.1, 8.6/8.2, 8.2/9.5, 12 (18) over 400, 500 8.8/8.8, 8.8/9.6; q16/kv1/hd96, 8
// (8) over 330, 470 7.9/6.9, 7.4/8.3; q48/kv3/hd256, 16 (48) over 400, 450 16.1/16.3, 16.3/18.1; q32/kv32/hd128, 2 (32) over 490, 590 8.1/8.1, 8.2/9.2; but
// q32/kv8/hd128, 16 (32) over 560, 610 9.8/8.6, 9.8/9.2, and with shared loads q24/kv1/hd128, 24 (36) over 630 10.5/9.1.
// f32 layers, four wavefronts a workgroup: a fourth page each is slower than the splits of up to 64 tiles, an eighth than those of 101 to 128, a tenth than those of
// up to 144. q32/kv8/hd128, 30 rows (64) over 190, 240, 290 11.7/12.3, 15.9/13.9, 16.1/13.8, 60 (120) over 310, 400, 480 17.0/15.2, 17.7/17.9, 18.0/19.2, 90 (184) over 710
// 28.3/24.9; q8/kv2/hd64, 30 (16) over 100 8.5/7.1; heads of 129 to 256 dims, q16/kv2/hd256, 24 (24) over 140 16.5/18.8.
// 1052 chunks of bf16 layers and 409 of f32 layers, 1 to 32 kv heads in groups of 1 to 16, at the lines and down to two thirds of them: 1.13 and 1.12 times as fast as
// split on the average, 0.96 at least. (With 26 + tiles / 2, 16 + tiles / 3 and 4 + tiles / 4 for all, some at the line took up to 1.23 times as long as split.)
bool whole_chunk(const Geom &g, size_t tiles, int n_pages, bool appends) {
    if (!may_stay_whole() || g.P > 256) return false;
    const size_t pages = (size_t)n_pages, per_head = tiles / (size_t)g.kv_heads; // tiles that walk the same pages
    if (g.f32) {
        if (g.P > 128 || (g.P > 64 && tiles <= 64 && pages > 12 && pages <= 16)) return false;
        if (g.P > 32 && tiles > 100 && tiles <= 144 && pages > (tiles <= 128 ? 28 : 36)) return false;
        return pages <= 4 + tiles / 4;
    }
    size_t line = g.P <= 128 ? 26 + tiles / 2 : 16 + tiles / 3;
    if (appends || per_head <= 4) {
        const bool near = g.kv_heads % 4 == 0;
        if (g.P <= 96 && (near || per_head <= 2)) line = g.kv_heads > 8 ? 26 + 2 * tiles / 5 : line;
        else if (g.P <= 96) line = g.P <= 32 ? 26 + tiles / 3 : g.P <= 64 ? 24 + tiles / 4 : 23 + tiles / 5;
        else if (g.P > 128) line = per_head == 1 ? std::min<size_t>(15 + tiles / 5, 18) : near ? 13 + tiles / 3 : 15 + tiles / 5;
        else if (near) line = per_head == 1 ? 27 : g.kv_heads > 8 ? 20 + 2 * tiles / 5 : 23 + tiles / 2;
        else line = per_head <= 2 ? 27 : g.kv_heads <= 2 ? 20 + tiles / 4 : 18 + tiles / 5;
    }
    return pages <= line;
}

hipStream_t as_stream(skv_stream s) { return reinterpret_cast<hipStream_t>(s); }

int32_t check_window(const skv_layer *L, size_t window_start) {
    if (L->len == 0) return fail(SKV_ERR_DIMENSION, "attention_decode sur KV vide");
    if (window_start >= L->len)
        return fail(SKV_ERR_DIMENSION, "attention_decode fenêtre vide: début=" +
                                           std::to_string(window_start) +
                                           ", len=" + std::to_string(L->len));
    if (L->g.ring_rows > 0 && window_start < L->floor_pos)
        return fail(SKV_ERR_DIMENSION,
                    "attention_decode: fenêtre début=" + std::to_string(window_start) +
                        " avant la plus ancienne ligne conservée " + std::to_string(L->floor_pos));
    return SKV_OK;
}

bool uses_flash(const skv_layer *L) { return skv_flag_flash_sdpa_enabled() && L->g.P <= 512; }
// The attention launch of a decode step can append the row itself: always on bf16 layers,
// on f32 layers where the f32 decode kernel serves the shape (head_dim up to 256, at most 16
// heads per group).
bool fused_append_built(const skv_layer *L) { return !L->g.f32 || (L->g.P <= 256 && L->g.gqa <= 16); }
// The fused pre-KV step is built for bf16 layers up to head_dim 512 and for f32 layers up to
// head_dim 256; wide f32 heads take the separate norm/rotation launches.
bool wide_f32_heads(const skv_layer *L) { return L->g.f32 && L->g.P > 256; }

// Pages that a launch of this window walks. ring: the layer is one, and has wrapped.
int pages_walked(const skv_layer *L, size_t window_start, bool ring) {
    return ring ? (int)std::min<size_t>((L->len + 15) / 16, (size_t)L->n_pages) : (int)((L->len + 15) / 16 - window_start / 16);
}

// Arguments of the matrix-core attention kernel for the layer's current length.
void fill_decode_args(const skv_layer *L, const float *q_dev, float *out_dev, size_t window_start,
                      const float *k_new, const float *v_new, size_t n_queries, size_t target_wgs,
                      DecodeArgs &a, bool keep_ring = false, bool whole_ok = false, int batch_wgs = 0) {
    Geom g = L->g;
    // A ring that has not wrapped is a full layer: every position in its own slot, no page but those in the queries' reach to walk and
    // no position to work out (512 rows of q16/kv8/hd256 on an empty ring of 1056 27.4 -> 23.2 us, over 512 38.6 -> 33.2, f32 over none
    // 66.5 -> 52.3; 256 rows of q32/kv8/hd128 over 700 25.9 -> 21.5).
    if (!keep_ring && L->len <= (size_t)g.ring_rows) g.ring_rows = 0;
    a.q = q_dev;
    a.out = out_dev;
    a.k_pool = L->k_pool;
    a.v_pool = L->v_pool;
    a.table = L->table_dev;
    a.part_o = L->part_o;
    a.part_m = L->part_m;
    a.part_l = L->part_l;
    a.len = (int)L->len;
    a.n_queries = (int)n_queries;
    a.q_pos0 = (int)(L->len - n_queries); // the queries are the last n_queries rows
    a.limit_cap = INT32_MAX;
    a.split_base = 0;
    a.window = n_queries > 1 ? (int)L->window : 0; // decode callers pass window_start themselves
    a.window_start = (int)window_start;
    a.n_pages = pages_walked(L, window_start, g.ring_rows > 0);
    if (g.ring_rows > 0) {
        a.page_first = 0;
        a.ring_t = (int)((L->len - 1) % (size_t)g.ring_rows);
        a.ring_base = (int)(L->len - 1) - a.ring_t;
    } else {
        a.page_first = (int)(window_start / 16);
    }
    a.waves = choose_waves(L, a.n_pages);
    a.splits = choose_splits(L, a.n_pages, L->len - window_start, a.waves, target_wgs);
    if (whole_ok && n_queries == 1 && a.n_pages <= whole_step_pages(g, batch_wgs)) {
        a.waves = 8;
        a.splits = 1;
    }
    a.splits_total = a.splits;
    // scores are multiplied by 1/sqrt(head_dim) (src/decode_resident/kernels.rs:36, 198, 395,
    // 575); log2(e) moves the softmax to base 2.
    a.qscale = (1.0f / std::sqrt((float)g.head_dim)) * 1.4426950408889634f;
    a.k_new = k_new;
    a.v_new = v_new;
    a.new_slot = (int)slot_of((long)L->len - 1, g.ring_rows);
    a.new_page = L->table[(size_t)(a.new_slot >> 4)];
    a.q_vec = (tuning().q_vec && (reinterpret_cast<uintptr_t>(q_dev) & 15) == 0 && (g.head_dim & 7) == 0) ? 1 : 0;
    a.g = g;
}

bool capturing(hipStream_t s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &status) != hipSuccess) {
        (void)hipGetLastError();
        return true; // what cannot be told is taken for the one that holds on to its scratch
    }
    return status != hipStreamCaptureStatusNone;
}

int32_t scratch_error(int status, size_t need) {
    if (status == StreamScratch::REFUSED)
        return fail(SKV_ERR_DEVICE, "prefill chunk: flux en capture, le tampon du flux est plus petit que les " +
                                        std::to_string(need) + " o requis (même appel d'abord hors capture)");
    return fail_hip((hipError_t)status, "prefill chunk: tampon des partiels");
}

// Split partials of a multi-query launch live in the context's scratch, grown on demand:
// [kv_heads][n_sets][n_queries * gqa] of (o[head_dim], m, l); in front of them `page_bytes` for
// pages of the chunk's own rows (*pages, a multiple of 256). The lease is the caller's until it has queued its launches.
int try_partials(skv_layer *L, hipStream_t s, size_t n_sets, size_t n_queries, DecodeArgs &a, StreamScratch::Lease &lease,
                 size_t page_bytes = 0, void **pages = nullptr, bool optional = false, size_t *asked = nullptr) {
    const Geom &g = L->g;
    const size_t n_part = (size_t)g.kv_heads * n_sets * n_queries * g.gqa;
    const size_t need = page_bytes + n_part * ((size_t)g.head_dim + 2) * sizeof(float);
    void *buf = nullptr;
    const int status = L->ctx->scratch.get(hip_scratch, s, need, capturing(s), lease, &buf, optional);
    if (asked) *asked = need;
    if (status != 0) return status;
    if (pages) *pages = buf;
    a.part_o = reinterpret_cast<float *>(static_cast<char *>(buf) + page_bytes);
    a.part_m = a.part_o + n_part * g.head_dim;
    a.part_l = a.part_m + n_part;
    return 0;
}
int32_t multi_query_partials(skv_layer *L, hipStream_t s, size_t n_sets, size_t n_queries, DecodeArgs &a,
                             StreamScratch::Lease &lease, size_t page_bytes = 0, void **pages = nullptr) {
    size_t need = 0;
    const int status = try_partials(L, s, n_sets, n_queries, a, lease, page_bytes, pages, false, &need);
    return status == 0 ? SKV_OK : scratch_error(status, need);
}

// The layer's pages as the queries of a chunk walk them: from position 0 on on a full layer, from
// position `lo` to the last row before `end` on a ring.
ChunkPages layer_pages(const Geom &g, size_t lo, size_t end) {
    ChunkPages c{};
    c.n_old = INT32_MAX;
    c.new_pos0 = INT32_MAX;
    if (g.ring_rows > 0) {
        c.n_old = lo < end ? (int)((end - 1) / 16 - lo / 16) + 1 : 0;
        c.first_pos = (int)(lo / 16 * 16);
        c.ring_pages = g.ring_rows / 16;
        c.start = (int)(lo / 16 % (size_t)c.ring_pages);
    }
    return c;
}

// The launch arguments that append n_rows rows at the layer's length.
AppendArgs append_args(const skv_layer *L, const float *k_dev, const float *v_dev, size_t n_rows) {
    AppendArgs a{};
    a.k_src = k_dev;
    a.v_src = v_dev;
    a.k_pool = L->k_pool;
    a.v_pool = L->v_pool;
    a.table = L->table_dev;
    a.first_pos = (long)L->len;
    a.n_rows = (int)n_rows;
    a.g = L->g;
    if (L->g.ring_rows > 0 && n_rows > (size_t)L->g.ring_rows) {
        // only the last ring_rows rows survive; skip the ones that would be overwritten
        const size_t skip = n_rows - (size_t)L->g.ring_rows;
        const size_t kv_dim = (size_t)L->g.kv_heads * L->g.head_dim;
        a.k_src += skip * kv_dim;
        a.v_src += skip * kv_dim;
        a.first_pos += (long)skip;
        a.n_rows = L->g.ring_rows;
    }
    return a;
}

// Whether a chunk on f32 pages has them split into terms by a launch of its own, once for all workgroups, instead of by each
// workgroup for its slots. That launch moves 10 bytes per value of the whole context (19 us at 4600 rows of 8 x 128) and stores
// the chunk's rows on the way; the attention behind it takes a quarter less on short walks and 5 to 10 % on long ones. So it pays
// where many slots share a page, and on rings, whose context is short and whose rows otherwise take a launch to pages of
// their own. Whole chunks on layers that are in no cache, in us, split by the workgroup / by a launch: q32/kv8/hd128, 512 rows over 0, 512,
// 1024, 2048, 4096 35.0/30.1, 57.8/50.3, 80.1/69.5, 113/107, 187/183, 256 rows (1024 slots) over 500, 2048, 8192 36.9/35.6, 62.8/64.2,
// 174/187, 64 rows over 8192 62.8/86.3; q28/kv4/hd128, 160 rows over 3000 54.7/56.9, 512 over 16000 587/540; q12/kv4/hd96, 512 rows
// (1536 slots) over 2000 50.4/50.9; q8/kv2/hd64, 512 rows over 2048, 4096 30.4/28.2, 42.5/39.3, 300 over 10000 55.1/56.8; q16/kv2/hd256,
// 128 rows (1024 slots) over 4096 71.1/70.2, 256 106/102, 512 188/173, over 16000 256 318/304; q16/kv8/hd256, 512 rows
// (1024 slots) over 1000 83.8/84.6. Rings: q16/kv8/hd256 of 1024 rows, 64, 256, 512, 1024 rows 62.6/58.6, 68.7/64.5, 77.0/76.9, 127/123;
// q32/kv8/hd128 of 512 rows, 64, 128 rows 32.3/28.9, 34.1/31.0, of 1024, 256, 512 48.4/44.4, 70.8/60.4; q8/kv2/hd64 of 1024, 128 rows 23.0/19.2.
bool f32_terms_pay(const Geom &g, size_t n_queries) {
    if (tuning().f32_terms != 1) return tuning().f32_terms > 1;
    return g.ring_rows > 0 || n_queries * (size_t)g.gqa >= (g.P > 128 ? 2048u : 1536u);
}

// Scratch for the terms of a chunk that walks `pairs` pairs of pages, of a layer of up to `layer_pairs`: the number of pairs it holds, 0 =
// none. A layer asks for all of its pairs at once while that is 128 MiB at most, then for twice as much each time, so that
// the chunks of a growing context seldom replace it. A quarter of what the chunk walks will do, the context is then taken in
// segments, each with partials of its own (four of them, 512 rows of q32/kv8/hd128 over 40000, cost 2 %; terms gain 5 to 10).
size_t terms_scratch(skv_layer *L, hipStream_t s, size_t pairs, size_t layer_pairs, StreamScratch::Lease &lease, void **terms) {
    const size_t one = f32_terms_bytes(L->g), limit = tuning().f32_terms_max, most = limit / one;
    size_t n = std::max<size_t>(((size_t)128 << 20) / one, 1);
    while (n < pairs) n *= 2;
    const size_t want = std::min(std::max(std::min(n, layer_pairs), pairs), most), least = (std::min(pairs, most) + 3) / 4;
    return want == 0 ? 0 : L->ctx->scratch.terms(hip_scratch, s, want * one, least * one, limit, lease, terms) / one;
}

// Such a chunk. Contexts of more pairs than the terms' scratch holds are taken in segments, each with
// splits of its own (512 rows of q32/kv8/hd128 over 16384, 40000, in us, segments of 128 MiB / 1 GiB 657/643, 1562/1532; over 8192,
// where two segments of 64 MiB take 357, one takes 340).
struct F32Plan {
    int first, last;    // pairs of entries of the page list
    int entries;        // of the list
    int segments, held; // pairs of a segment
    int splits;         // of a segment
    bool halves;
    int sets() const { return segments * splits; }
};
// walked: pages that a workgroup walks of all segments; most: pairs that the scratch holds
F32Plan plan_f32_chunk(const Geom &g, size_t n_queries, int first_entry, int entries, int walked, int max_splits, size_t most) {
    F32Plan p{};
    p.first = first_entry / 2;
    p.last = (entries + 1) / 2;
    p.entries = entries;
    const size_t pairs = (size_t)(p.last - p.first);
    p.segments = (int)((pairs + most - 1) / most);
    p.held = (int)((pairs + (size_t)p.segments - 1) / (size_t)p.segments);
    // Halves cover half the slots and walk two pairs at a time: the same time per workgroup with half as many splits, so fewer
    // partials, but they copy each page for half as many slots, which costs more on long walks. Whole chunks, one tile / halves, in us: q32/kv8/hd128, 512 rows
    // over 0, 512, 1024, 2048, 6000, 8192, 16384 (two splits / one) 41.1/30.0, 58.4/50.1, 74.5/69.3, 111/106, 254/254, 333/336, 627/642; q8/kv2/hd64,
    // 512 rows over 2048, 4096, 10000 (eight / four) 32.6/28.1, 43.0/39.1, 73.4/72.2, 448 over 1856, 3420 (nine / four) 31.1/26.5, 39.8/34.7; but
    // q28/kv4/hd128, 300 rows over 3000 (three / one) 90.9/114. So a ninth of the workgroups may go.
    const size_t pages = (size_t)walked / (size_t)p.segments;
    const int one = chunk_splits(g, n_queries, (size_t)f32_prefill_slots(g.P, false), pages);
    const int two = chunk_splits(g, n_queries, (size_t)f32_prefill_slots(g.P, true), pages);
    p.halves = g.P <= 128 && tuning().prefill_tiles2_min_pages < 0 && 18 * two >= 8 * one && walked <= 300;
    // (choose_splits' number, which the split knobs of decode launches bound, is the larger one unless they do)
    p.splits = std::min(max_splits, p.halves ? two : one);
    return p;
}
int32_t run_f32_chunk(const F32Plan &p, DecodeArgs a, const ChunkPages &pages, void *terms, int pos_lo, const float *k_new,
                      const float *v_new, hipStream_t s, bool merge = true) {
    a.splits = p.splits;
    a.splits_total = p.sets();
    a.k_new = a.v_new = nullptr;
    for (int seg = 0; seg < p.segments; ++seg) {
        TermPairs t;
        t.terms = terms;
        t.first = p.first + seg * p.held;
        t.held = std::min(p.held, p.last - t.first);
        t.entries = p.entries;
        t.pos_lo = pos_lo;
        t.pos_hi = a.q_pos0 + a.n_queries - 1;
        t.k_src = k_new;
        t.v_src = v_new;
        t.new_pos = k_new ? a.q_pos0 : INT32_MAX;
        t.vec = k_new && (reinterpret_cast<uintptr_t>(k_new) & 15) == 0 && a.g.head_dim % 4 == 0;
        a.split_base = seg * p.splits;
        SKV_HIP(launch_f32_terms(a, pages, t, s));
        SKV_HIP(launch_f32_prefill(a, pages, &t, p.halves, s));
    }
    if (merge && a.splits_total > 1) SKV_HIP(launch_merge_rows(a, s));
    return SKV_OK;
}

// k_new / v_new non-null: the row at position len-1 has not been written yet and the
// attention kernel appends it itself (the host bookkeeping has already advanced).
// n_queries > 1: chunked prefill over the cache; the last n_queries rows are the new ones
// and query i attends positions up to len - n_queries + i, each through the layer's
// sliding window. The matrix-core kernel only.
// attn_scalar > 0 replaces head_dim under the square root of the score scale
// (encode_query_attention_scale, src/decode_resident/layers.rs:7-33); pre non-null asks the
// kernel to norm and rotate q and the new k row itself.
struct PreKv {
    const float *rope;
    const float *q_norm_w;
    const float *k_norm_w;
    float eps;
    int rope_dims;
    int rope_style;
    const float *gate;  // multiplied into the context through a sigmoid (null = none)
    int q_head_stride;  // elements between the heads of q and of gate (0 = head_dim)
};

// Points the launch's split partials at `buf` instead of the layer's own buffers
// (decode, one query row): [kv_heads][splits][gqa] of (o[head_dim], m, l).
int32_t partials_in(void *buf, size_t buf_bytes, DecodeArgs &a) {
    const Geom &g = a.g;
    const size_t n_part = (size_t)g.kv_heads * (size_t)a.splits_total * (size_t)g.gqa * (size_t)a.n_queries;
    const size_t need = n_part * ((size_t)g.head_dim + 2) * sizeof(float);
    if (need > buf_bytes)
        return fail(SKV_ERR_DIMENSION, "decode_step_static: partiels split-K de " + std::to_string(need) +
                                           " o > tampon statique de " + std::to_string(buf_bytes) + " o");
    a.part_o = reinterpret_cast<float *>(buf);
    a.part_m = a.part_o + n_part * g.head_dim;
    a.part_l = a.part_m + n_part;
    return SKV_OK;
}

int32_t encode_attention(skv_layer *L, hipStream_t s, const float *q_dev, float *out_dev,
                         size_t window_start, const float *k_new = nullptr,
                         const float *v_new = nullptr, size_t n_queries = 1,
                         float attn_scalar = 0.0f, const PreKv *pre = nullptr,
                         void *static_partials = nullptr) {
    int32_t rc = check_window(L, window_start);
    if (rc) return rc;
    const Geom &g = L->g;
    if (static_partials && (n_queries != 1 || !uses_flash(L)))
        return fail(SKV_ERR_CONFIG, "decode_step_static: une ligne de requête, noyau matriciel seulement");
    StreamScratch::Lease lease;
    // Whether the context lies over what other workgroups read: the queries (and the gate between them), a step's new row. (A chunk's
    // rows are stored by a launch in front, or the caller has looked.)
    const bool over = over_queries(g, out_dev, q_dev, n_queries, pre ? (size_t)pre->q_head_stride : 0) ||
                      (n_queries == 1 && (over_rows(g, out_dev, k_new, 1) || over_rows(g, out_dev, v_new, 1)));
    // Such a context of an unsplit launch, and a gated one of any (the merge reads the gate), is written aside and copied behind the launch.
    float *aside = nullptr;
    const auto place = [&](int splits, float *&out, bool late = false) -> int32_t {
        if (!(over || late) || (splits > 1 && !(pre && pre->gate))) return SKV_OK;
        if (n_queries == 1) {
            aside = L->out_stage;
        } else {
            void *buf = nullptr;
            const size_t need = n_queries * (size_t)g.q_heads * g.head_dim * sizeof(float);
            const int status = L->ctx->scratch.get(hip_scratch, s, need, capturing(s), lease, &buf);
            if (status != 0) return scratch_error(status, need);
            aside = static_cast<float *>(buf);
        }
        out = aside;
        return SKV_OK;
    };
    const auto settle = [&]() -> int32_t {
        if (aside) SKV_HIP(launch_copy(out_dev, aside, n_queries * (size_t)g.q_heads * g.head_dim, s));
        return SKV_OK;
    };
    if (g.f32 && (uses_flash(L) || n_queries > 1)) {
        // the f32 element's matrix kernels: 16 query slots per workgroup, the context split while
        // that leaves compute units idle; one query row of narrow heads takes the kernel that
        // can append the row (and norm and rotate q and k) itself
        DecodeArgs a{};
        fill_decode_args(L, q_dev, out_dev, window_start, k_new, v_new, n_queries, decode_target_wgs(), a);
        if ((k_new || v_new || pre) && n_queries == 1 && !f32_decode_kernel_serves(a))
            return fail(SKV_ERR_CONFIG, "KV f32: étape fusionnée non construite pour cette forme");
        if (pre) {
            a.pre = 1;
            a.rope = pre->rope;
            a.q_norm_w = pre->q_norm_w;
            a.k_norm_w = pre->k_norm_w;
            a.eps = pre->eps;
            a.rope_dims = pre->rope ? pre->rope_dims : 0;
            a.rope_style = pre->rope_style;
            a.gate = pre->gate;
            a.q_head_stride = pre->q_head_stride;
        }
        if (attn_scalar > 0.0f) a.qscale = (1.0f / std::sqrt(attn_scalar)) * 1.4426950408889634f;
        const bool by_terms = n_queries > 1 && takes_f32_chunk_kernel(g, n_queries, (size_t)a.n_pages);
        const auto store_rows = [&]() -> int32_t { // rows that the terms' launch would have stored
            if (n_queries == 1 || !k_new) return SKV_OK;
            AppendArgs w = append_args(L, k_new, v_new, n_queries);
            w.first_pos -= (long)n_queries; // (counted already)
            SKV_HIP(launch_append(w, s));
            a.k_new = a.v_new = nullptr;
            return SKV_OK;
        };
        if (by_terms) {
            const size_t lo = std::max(window_start, skv_window_start(L->len - n_queries, L->window));
            const ChunkPages pages = layer_pages(a.g, lo, L->len); // (a ring's list begins at `lo`, a full layer's at 0)
            // (a captured launch makes no terms: their scratch is replaced and dropped)
            if (f32_terms_pay(a.g, n_queries) && !capturing(s)) {
                const bool ring = a.g.ring_rows > 0;
                const int first = ring ? 0 : (int)(lo / 16), entries = ring ? pages.n_old : a.page_first + a.n_pages;
                StreamScratch::Lease terms_lease;
                void *terms = nullptr;
                const size_t most = terms_scratch(L, s, (size_t)((entries + 1) / 2 - first / 2), (size_t)(L->n_pages + 1) / 2, terms_lease, &terms);
                if (most > 0) {
                    const F32Plan plan = plan_f32_chunk(g, n_queries, first, entries, ring ? entries : a.n_pages, a.splits, most);
                    DecodeArgs b = a;
                    b.splits_total = plan.sets();
                    if (plan.sets() == 1 || try_partials(L, s, (size_t)plan.sets(), n_queries, b, lease, 0, nullptr, true) == 0) {
                        rc = place(plan.sets(), b.out, reads_again(g, out_dev, q_dev));
                        if (!rc) rc = run_f32_chunk(plan, b, pages, terms, (int)lo, k_new, v_new, s);
                        return rc ? rc : settle();
                    }
                }
                // no memory for them: the other way needs none
            }
            rc = store_rows();
            if (rc) return rc;
            const bool halves = f32_halves(g, n_queries * (size_t)g.gqa, (size_t)a.n_pages);
            // (choose_splits' number, which the split knobs of decode launches bound, is the larger one unless they do)
            a.splits = std::min(a.splits, chunk_splits(g, n_queries, (size_t)f32_prefill_slots(g.P, halves), (size_t)a.n_pages));
            a.splits_total = a.splits;
            if (a.splits > 1) {
                int32_t rc2 = multi_query_partials(L, s, (size_t)a.splits, n_queries, a, lease);
                if (rc2) return rc2;
            }
            rc = place(a.splits, a.out, reads_again(g, out_dev, q_dev));
            if (rc) return rc;
            SKV_HIP(launch_f32_prefill(a, pages, nullptr, halves, s));
            if (a.splits > 1) SKV_HIP(launch_merge_rows(a, s));
            return settle();
        }
        if (n_queries > 1) {
            rc = store_rows(); // (a knob that turned between the caller's look at it and this one)
            if (rc) return rc;
            const size_t tiles = (n_queries * (size_t)g.gqa + 15) / 16 * (size_t)g.kv_heads;
            size_t want = std::max<size_t>(2 * decode_target_wgs() / tiles, 1);
            // a chunk that a ring holds without wrapping: whole eights of pages a split (130 rows of q16/kv8/hd256 on an empty
            // ring: 22.3 us with one, 29.7 with two and a merge)
            if (L->g.ring_rows > 0) want = std::min(want, std::max<size_t>((size_t)a.n_pages / 8, 1));
            a.splits = (int)std::min<size_t>((size_t)a.splits, want);
            if (tiles > (size_t)g.kv_heads) a.splits = xcd_splits(a.splits, g.kv_heads, a.n_pages, 4, 16);
            if (!over && whole_chunk(g, tiles, a.n_pages, false)) a.splits = 1;
            a.splits_total = a.splits;
            if (a.splits > 1) {
                int32_t rc2 = multi_query_partials(L, s, (size_t)a.splits, n_queries, a, lease);
                if (rc2) return rc2;
            }
        }
        if (static_partials && a.splits > 1) {
            int32_t rc2 = partials_in(static_partials, SKV_STATIC_SCRATCH_BYTES, a);
            if (rc2) return rc2;
        }
        rc = place(a.splits, a.out);
        if (rc) return rc;
        SKV_HIP(launch_f32_split(a, s));
        if (a.splits > 1) SKV_HIP(n_queries > 1 ? launch_merge_rows(a, s) : launch_merge(a, s));
        return settle();
    }
    const bool use_flash = uses_flash(L) || n_queries > 1;
    if (!use_flash) {
        const size_t need = (size_t)g.q_heads * L->capacity;
        if (L->scores_cap < need) {
            if (L->scores) {
                SKV_HIP(hipDeviceSynchronize());
                SKV_HIP(hipFree(L->scores));
                L->scores = nullptr;
                L->scores_cap = 0;
            }
            SKV_HIP(hipMalloc(&L->scores, need * sizeof(float)));
            L->scores_cap = need;
        }
        NaiveArgs a{};
        a.q = q_dev;
        a.out = out_dev;
        a.k_pool = L->k_pool;
        a.v_pool = L->v_pool;
        a.table = L->table_dev;
        a.scores = L->scores;
        a.len = (long)L->len;
        a.window_start = (long)window_start;
        a.inv_scale = 1.0f / std::sqrt(attn_scalar > 0.0f ? attn_scalar : (float)g.head_dim);
        a.g = g;
        rc = place(1, a.out);
        if (rc) return rc;
        SKV_HIP(launch_naive(a, s));
        return settle();
    }
    DecodeArgs a{};
    fill_decode_args(L, q_dev, out_dev, window_start, k_new, v_new, n_queries, decode_target_wgs(), a, false, !over);
    if (attn_scalar > 0.0f) a.qscale = (1.0f / std::sqrt(attn_scalar)) * 1.4426950408889634f;
    if (pre) {
        a.pre = 1;
        a.rope = pre->rope;
        a.q_norm_w = pre->q_norm_w;
        a.k_norm_w = pre->k_norm_w;
        a.eps = pre->eps;
        a.rope_dims = pre->rope ? pre->rope_dims : 0;
        a.rope_style = pre->rope_style;
        a.gate = pre->gate;
        a.q_head_stride = pre->q_head_stride;
    }
    const bool use_tiles = n_queries > 1 && takes_tile_kernel(a.g, n_queries, (size_t)a.n_pages);
    TileShape shape = TileShape::one_tile;
    if (n_queries > 1) {
        // split the context only while the query tiles alone leave compute units idle, and
        // keep the partials in the context's scratch
        shape = prefill_shape(g, n_queries * (size_t)g.gqa, (size_t)a.n_pages);
        if (!use_tiles && g.P <= 256 && tuning().forced_waves == 0) {
            // eight wavefronts, one page each before the context is split; four where the slot tiles
            // alone are two workgroups and more for every compute unit and narrow enough that it holds
            // several (256 rows of q32/kv8/hd128 over 0, 1024 rows: 11.7/24.1 us with four, 14.1/24.4 with
            // eight; 256 rows of q16/kv2/hd256: 14.2/30.1 and 13.5/24.6)
            const size_t slot_tiles = (n_queries * (size_t)g.gqa + 15) / 16 * (size_t)g.kv_heads;
            a.waves = g.P <= 128 && slot_tiles >= 512 ? 4 : 8;
            a.splits = choose_splits(L, a.n_pages, L->len - window_start, a.waves, decode_target_wgs());
        }
        const size_t per_wg = use_tiles ? (size_t)prefill_tile_slots(g.P, shape) : 16;
        const size_t tiles = (n_queries * (size_t)g.gqa + per_wg - 1) / per_wg * (size_t)g.kv_heads;
        size_t want = std::max<size_t>((use_tiles ? tuning().prefill_wgs : 256) / tiles, 1);
        if (use_tiles) {
            want = std::min<size_t>(want, std::max<size_t>((size_t)a.n_pages / 16, 1));
            want = std::min<size_t>(want, tuning().prefill_max_splits);
        }
        a.splits = (int)std::min<size_t>((size_t)a.splits, want);
        if (!use_tiles && tiles > (size_t)g.kv_heads) a.splits = xcd_splits(a.splits, g.kv_heads, a.n_pages, a.waves, 10);
        if (!use_tiles && !over && whole_chunk(g, tiles, a.n_pages, k_new != nullptr)) a.splits = 1;
        a.splits_total = a.splits;
        if (a.splits > 1) {
            int32_t rc2 = multi_query_partials(L, s, (size_t)a.splits, n_queries, a, lease);
            if (rc2) return rc2;
        }
    }
    if (static_partials && a.splits_total > 1) {
        int32_t rc2 = partials_in(static_partials, SKV_STATIC_SCRATCH_BYTES, a);
        if (rc2) return rc2;
    }
    rc = place(a.splits, a.out);
    if (rc) return rc;
    if (use_tiles) {
        const size_t lo = std::max(window_start, skv_window_start(L->len - n_queries, L->window));
        SKV_HIP(launch_prefill_tiles(a, layer_pages(a.g, lo, L->len), shape, s));
        if (a.splits > 1) SKV_HIP(launch_merge_rows(a, s));
    } else {
        SKV_HIP(launch_decode(a, s));
    }
    return settle();
}

void appended(skv_layer *L, size_t n_rows) {
    L->len += n_rows;
    if (L->g.ring_rows > 0 && L->len > (size_t)L->g.ring_rows)
        L->floor_pos = std::max(L->floor_pos, L->len - (size_t)L->g.ring_rows);
}

// A layer that counts n rows ahead of the launch that writes them, until the end of the scope unless they are written by
// then: an error, or an exception on the way (a launch's scratch may have to grow), leaves it as it was.
struct RowsAhead {
    skv_layer *L;
    size_t n;
    bool written = false;
    RowsAhead(skv_layer *layer, size_t rows) : L(layer), n(rows) { L->len += n; }
    RowsAhead(const RowsAhead &) = delete;
    ~RowsAhead() {
        if (!written) L->len -= n;
    }
};

int32_t encode_append(skv_layer *L, hipStream_t s, const float *k_dev, const float *v_dev,
                      size_t n_rows) {
    if (n_rows == 0) return SKV_OK;
    if (L->len + n_rows > L->capacity)
        return fail(SKV_ERR_DIMENSION, "append KV résident: capacité " +
                                           std::to_string(L->capacity) + " atteinte (overflow)");
    SKV_HIP(launch_append(append_args(L, k_dev, v_dev, n_rows), s));
    appended(L, n_rows);
    return SKV_OK;
}

} // namespace

extern "C" {

const char *skv_last_error(void) { return g_last_error.c_str(); }
int32_t skv_abi_version(void) { return 1; }

int32_t skv_ctx_create(int32_t device, skv_ctx **out) try {
    if (!out) return fail(SKV_ERR_DEVICE, "skv_ctx_create: out nul");
    *out = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count <= 0)
        return fail(SKV_ERR_DEVICE, "aucun GPU HIP disponible (le chemin KV gfx950 exige un MI355X)");
    if (device < 0 || device >= count)
        return fail(SKV_ERR_CONFIG, "device " + std::to_string(device) + " hors plage");
    SKV_HIP(hipSetDevice(device));
    // The synchronous host entry points run on the legacy default stream, which
    // orders itself against every blocking stream of the process (a framework's
    // default stream included), so a host call that follows device-side calls on
    // such a stream sees their effect without an explicit wait.
    // the library's set-up call on this device: the address of the static scratch array here
    void *static_scratch = nullptr;
    SKV_HIP(static_scratch_ptr(device, &static_scratch));
    skv_ctx *c = new skv_ctx();
    c->device = device;
    c->stream = nullptr;
    c->static_scratch = static_scratch;
    c->arena_cap = env_usize("SKV_ARENA_MAX_MB", 4096) << 20;
    *out = c;
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

void skv_ctx_destroy(skv_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    (void)hipDeviceSynchronize();
    {
        std::lock_guard<std::mutex> lk(ctx->arena_mu);
        ctx->closed = true;
    }
    ctx_drain(ctx);
    ctx_release(ctx);
}

int32_t skv_ctx_synchronize(skv_ctx *ctx) try {
    if (!ctx) return fail(SKV_ERR_DEVICE, "ctx nul");
    SKV_HIP(hipSetDevice(ctx->device));
    SKV_HIP(hipDeviceSynchronize());
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

void skv_layer_destroy(skv_layer *L) {
    if (!L) return;
    (void)hipSetDevice(L->ctx->device);
    (void)hipDeviceSynchronize();
    for (auto &b : L->leased) arena_put(L->ctx, b.first, b.second);
    if (L->scores) (void)hipFree(L->scores);
    delete L;
}

// Shape checks of full_attention_with_element (src/decode_resident/attention.rs:56-108) and
// the geometry, page count and buffer sizes that follow from them; shared by the factory and
// by skv_layer_bytes so that the budget figure is the factory's own arithmetic.
struct LayerPlan {
    Geom g{};
    int n_pages = 0;
    int max_splits = 1;
    size_t pool_bytes = 0, table_bytes = 0, part_o_bytes = 0, part_ml_bytes = 0, q_bytes = 0, kv_stage_bytes = 0;
    size_t total() const {
        // every buffer is its own allocation, rounded up by the allocator to 256 bytes at least
        auto r = [](size_t b) { return (std::max<size_t>(b, 256) + 255) / 256 * 256; };
        return 2 * r(pool_bytes) + r(table_bytes) + r(part_o_bytes) + 2 * r(part_ml_bytes) + 2 * r(q_bytes) +
               r(kv_stage_bytes);
    }
};

// rollback_rows: rows a ring layer keeps behind its window (SIZE_MAX = the default: the
// environment's SKV_RING_SLACK_ROWS, else 32)
static int32_t plan_layer(size_t capacity, size_t q_heads, size_t kv_heads, size_t head_dim, int32_t dtype,
                          size_t window, size_t rollback_rows, LayerPlan &p) {
    if (capacity == 0 || q_heads == 0 || kv_heads == 0 || head_dim == 0)
        return fail(SKV_ERR_CONFIG, "FullAttentionMetalState: dimension nulle");
    if (q_heads % kv_heads != 0)
        return fail(SKV_ERR_CONFIG, "GQA invalide: q_heads=" + std::to_string(q_heads) +
                                        " non multiple de kv_heads=" + std::to_string(kv_heads));
    if (dtype != SKV_DTYPE_BF16 && dtype != SKV_DTYPE_F32)
        return fail(SKV_ERR_CONFIG, "élément KV inconnu: " + std::to_string(dtype));
    const bool f32 = dtype == SKV_DTYPE_F32;
    const int P = padded_head_dim(head_dim);
    if (P == 0) return fail(SKV_ERR_CONFIG, "head_dim > 512 non supporté");
    if (capacity > (size_t)1 << 30 || q_heads > 4096 || kv_heads > 4096 || window > (size_t)1 << 30 ||
        (rollback_rows != SIZE_MAX && rollback_rows > (size_t)1 << 30))
        return fail(SKV_ERR_CONFIG, "capacité KV déborde");
    Geom &g = p.g;
    g.q_heads = (int)q_heads;
    g.kv_heads = (int)kv_heads;
    g.head_dim = (int)head_dim;
    g.P = P;
    set_gqa(g);
    g.f32 = f32 ? 1 : 0;
    g.tile_elems = P * 16 * (f32 ? 2 : 1);
    g.page_elems = (int)kv_heads * g.tile_elems;
    size_t rows = capacity;
    if (window > 0) {
        // The ring keeps the window plus some rows behind it, so that the rows a speculative
        // verify appended can be rolled back (truncate) without the ring having overwritten
        // what the next query attends: the reference keeps the whole cache and rolls back
        // freely (src/decoder/attention_cache.rs:72-100). A ring never needs more rows than
        // the capacity.
        const size_t slack = rollback_rows != SIZE_MAX ? rollback_rows : env_usize("SKV_RING_SLACK_ROWS", 32);
        size_t ring = (window + slack + 15) / 16 * 16;
        ring = std::min(ring, (capacity + 15) / 16 * 16);
        g.ring_rows = (int)ring;
        rows = ring;
    }
    p.n_pages = (int)((rows + 15) / 16);
    p.pool_bytes = (size_t)p.n_pages * kv_heads * pool_head_dim(head_dim) * 16 * (f32 ? sizeof(float) : sizeof(uint16_t));
    p.max_splits = std::min(decode_max_splits(), std::max(1, p.n_pages));
    const size_t n_part = (size_t)kv_heads * p.max_splits * g.gqa;
    p.table_bytes = (size_t)p.n_pages * sizeof(int32_t);
    p.part_o_bytes = n_part * head_dim * sizeof(float);
    p.part_ml_bytes = n_part * sizeof(float);
    p.q_bytes = q_heads * head_dim * sizeof(float);
    p.kv_stage_bytes = 2 * kv_heads * head_dim * sizeof(float);
    return SKV_OK;
}

int32_t skv_layer_bytes(size_t capacity, size_t q_heads, size_t kv_heads, size_t head_dim, int32_t dtype,
                        size_t window, uint64_t *bytes) try {
    if (!bytes) return fail(SKV_ERR_DEVICE, "skv_layer_bytes: pointeur nul");
    LayerPlan p;
    int32_t rc = plan_layer(capacity, q_heads, kv_heads, head_dim, dtype, window, SIZE_MAX, p);
    if (rc) return rc;
    *bytes = (uint64_t)p.total();
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_check_allocation(skv_ctx *ctx, uint64_t requested, uint64_t static_cap, uint64_t headroom,
                             uint64_t *available, uint64_t *projected) try {
    if (!ctx) return fail(SKV_ERR_DEVICE, "skv_check_allocation: ctx nul");
    SKV_HIP(hipSetDevice(ctx->device));
    size_t free_b = 0, total_b = 0;
    SKV_HIP(hipMemGetInfo(&free_b, &total_b));
    // effective_limit: the smallest of the caps that are set (src/memory_guard.rs:109-127); the
    // device's memory minus the headroom stands where the host's memory stands there
    uint64_t limit = (uint64_t)total_b > headroom ? (uint64_t)total_b - headroom : 0;
    if (static_cap) limit = std::min(limit, static_cap);
    // what the context's arena holds is free for the next layers of the same context
    uint64_t held = 0;
    {
        std::lock_guard<std::mutex> lk(ctx->arena_mu);
        held = ctx->arena_bytes;
    }
    const uint64_t used = (uint64_t)(total_b - free_b);
    const uint64_t current = used > held ? used - held : 0;
    uint64_t proj = 0, avail = 0;
    const int32_t over = skv_memory_projection(current, 0, requested, limit, &proj, &avail);
    if (available) *available = avail;
    if (projected) *projected = proj;
    if (over)
        return fail(SKV_ERR_MEMORY, "garde mémoire: demande " + std::to_string(requested) + " o, projection " +
                                        std::to_string(proj) + " o > plafond " + std::to_string(limit) +
                                        " o (disponible " + std::to_string(avail) + " o)");
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_layer_create(skv_ctx *ctx, size_t capacity, size_t q_heads, size_t kv_heads,
                         size_t head_dim, int32_t dtype, size_t window, skv_layer **out) {
    return skv_layer_create_ring(ctx, capacity, q_heads, kv_heads, head_dim, dtype, window, SIZE_MAX, out);
}

int32_t skv_layer_bytes_ring(size_t capacity, size_t q_heads, size_t kv_heads, size_t head_dim, int32_t dtype,
                             size_t window, size_t rollback_rows, uint64_t *bytes) try {
    if (!bytes) return fail(SKV_ERR_DEVICE, "skv_layer_bytes: pointeur nul");
    LayerPlan p;
    int32_t rc = plan_layer(capacity, q_heads, kv_heads, head_dim, dtype, window, rollback_rows, p);
    if (rc) return rc;
    *bytes = (uint64_t)p.total();
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_layer_create_ring(skv_ctx *ctx, size_t capacity, size_t q_heads, size_t kv_heads, size_t head_dim,
                              int32_t dtype, size_t window, size_t rollback_rows, skv_layer **out) try {
    if (!ctx || !out) return fail(SKV_ERR_DEVICE, "skv_layer_create: pointeur nul");
    *out = nullptr;
    LayerPlan plan;
    {
        int32_t rc = plan_layer(capacity, q_heads, kv_heads, head_dim, dtype, window, rollback_rows, plan);
        if (rc) return rc;
    }
    SKV_HIP(hipSetDevice(ctx->device));

    skv_layer *L = new skv_layer();
    L->ctx = ctx;
    L->capacity = capacity;
    L->window = window;
    L->g = plan.g;
    const Geom &g = L->g;
    L->n_pages = plan.n_pages;
    const size_t pool_bytes = plan.pool_bytes;
    const size_t q_dim = q_heads * head_dim;
    const size_t kv_dim = kv_heads * head_dim;
    L->max_splits = plan.max_splits;
    const size_t n_part = (size_t)kv_heads * L->max_splits * g.gqa;

    hipError_t e = hipSuccess;
    auto alloc = [&](void **p, size_t bytes) {
        if (e != hipSuccess) return;
        size_t got = 0;
        e = arena_get(ctx, bytes, p, &got);
        if (e == hipSuccess) L->leased.emplace_back(*p, got);
    };
    alloc((void **)&L->k_pool, pool_bytes);
    alloc((void **)&L->v_pool, pool_bytes);
    alloc((void **)&L->table_dev, (size_t)L->n_pages * sizeof(int32_t));
    alloc((void **)&L->part_o, n_part * head_dim * sizeof(float));
    alloc((void **)&L->part_m, n_part * sizeof(float));
    alloc((void **)&L->part_l, n_part * sizeof(float));
    alloc((void **)&L->q_stage, q_dim * sizeof(float));
    alloc((void **)&L->out_stage, q_dim * sizeof(float));
    alloc((void **)&L->kv_stage, 2 * kv_dim * sizeof(float));
    // Padding dims and rows past `len` are multiplied by zero probabilities and zero
    // query padding; they must hold finite values, so the pools start at zero.
    if (e == hipSuccess) e = hipMemsetAsync(L->k_pool, 0, pool_bytes, ctx->stream);
    if (e == hipSuccess) e = hipMemsetAsync(L->v_pool, 0, pool_bytes, ctx->stream);
    L->table.resize(L->n_pages);
    for (int i = 0; i < L->n_pages; ++i) L->table[i] = i;
    if (e == hipSuccess) e = launch_iota(L->table_dev, L->n_pages, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        skv_layer_destroy(L);
        return fail_hip(e, "allocation du cache KV");
    }
    *out = L;
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_layer_create_for(skv_ctx *ctx, size_t capacity, size_t q_heads, size_t kv_heads,
                             size_t head_dim, int32_t sampled, skv_layer **out) try {
    const int32_t dtype = skv_flag_kv_bf16_for(sampled) ? SKV_DTYPE_BF16 : SKV_DTYPE_F32;
    return skv_layer_create(ctx, capacity, q_heads, kv_heads, head_dim, dtype, 0, out);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_layer_set_block_table(skv_layer *L, const int32_t *table, size_t n) try {
    if (!L || !table) return fail(SKV_ERR_DEVICE, "set_block_table: pointeur nul");
    if (L->len != 0) return fail(SKV_ERR_DIMENSION, "set_block_table: cache non vide");
    if (n != (size_t)L->n_pages)
        return fail(SKV_ERR_DIMENSION, "set_block_table: attendu " + std::to_string(L->n_pages) +
                                           " entrées, reçu " + std::to_string(n));
    std::vector<char> seen(n, 0);
    for (size_t i = 0; i < n; ++i) {
        if (table[i] < 0 || (size_t)table[i] >= n || seen[table[i]])
            return fail(SKV_ERR_DIMENSION, "set_block_table: pas une permutation");
        seen[table[i]] = 1;
    }
    SKV_HIP(hipSetDevice(L->ctx->device));
    L->table.assign(table, table + n);
    SKV_HIP(hipMemcpyAsync(L->table_dev, L->table.data(), n * sizeof(int32_t), hipMemcpyHostToDevice,
                           L->ctx->stream));
    SKV_HIP(hipStreamSynchronize(L->ctx->stream));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

size_t skv_layer_pages(const skv_layer *L) { return L ? (size_t)L->n_pages : 0; }
size_t skv_kv_dim(const skv_layer *L) { return L ? (size_t)L->g.kv_heads * L->g.head_dim : 0; }
size_t skv_len(const skv_layer *L) { return L ? L->len : 0; }
size_t skv_capacity(const skv_layer *L) { return L ? L->capacity : 0; }
size_t skv_q_heads(const skv_layer *L) { return L ? (size_t)L->g.q_heads : 0; }
size_t skv_kv_heads(const skv_layer *L) { return L ? (size_t)L->g.kv_heads : 0; }
size_t skv_head_dim(const skv_layer *L) { return L ? (size_t)L->g.head_dim : 0; }
size_t skv_window(const skv_layer *L) { return L ? L->window : 0; }
size_t skv_logical_byte_len(const skv_layer *L) {
    return L ? L->capacity * (size_t)L->g.kv_heads * L->g.head_dim * (L->g.f32 ? 4 : 2) : 0;
}

int32_t skv_truncate(skv_layer *L, size_t len) try {
    if (!L) return fail(SKV_ERR_DEVICE, "truncate: pointeur nul");
    if (len > L->capacity)
        return fail(SKV_ERR_DIMENSION, "truncate KV " + std::to_string(len) + " > capacité " +
                                           std::to_string(L->capacity));
    L->len = len;
    if (len == 0) L->floor_pos = 0;
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_seed(skv_layer *L, const float *keys, const float *values, size_t n_elems,
                 size_t n_rows) try {
    if (!L) return fail(SKV_ERR_DEVICE, "seed: pointeur nul");
    if (n_rows > L->capacity)
        return fail(SKV_ERR_DIMENSION, "seed KV " + std::to_string(n_rows) + " > capacité " +
                                           std::to_string(L->capacity));
    const size_t kv_dim = skv_kv_dim(L);
    const size_t expected = n_rows * kv_dim;
    if (n_elems != expected)
        return fail(SKV_ERR_DIMENSION, "seed KV: attendu " + std::to_string(expected) + " (=" +
                                           std::to_string(n_rows) + "×" + std::to_string(kv_dim) +
                                           "), reçu " + std::to_string(n_elems));
    if (n_rows > 0 && (!keys || !values)) return fail(SKV_ERR_DEVICE, "seed: pointeur nul");
    SKV_HIP(hipSetDevice(L->ctx->device));
    L->len = 0;
    L->floor_pos = 0;
    if (n_rows == 0) return SKV_OK;
    hipStream_t s = L->ctx->stream;
    // RETI_RUST_KV_BF16_SIM_KONLY / _VONLY (src/decode_resident/attention.rs:573-585): on an
    // f32 cache the seed keeps K alone, or else V alone, at bf16 precision (still stored as f32)
    std::vector<float> rounded;
    if (L->g.f32 && (skv_flag_kv_bf16_sim_konly() || skv_flag_kv_bf16_sim_vonly())) {
        const bool k_only = skv_flag_kv_bf16_sim_konly() != 0; // K wins when both are set, as in the match
        const float *src = k_only ? keys : values;
        rounded.resize(expected);
        for (size_t i = 0; i < expected; ++i) {
            const uint32_t b = (uint32_t)skv_f32_to_bf16_bits(src[i]) << 16;
            std::memcpy(&rounded[i], &b, sizeof(float));
        }
        (k_only ? keys : values) = rounded.data();
    }
    float *stage = nullptr;
    SKV_HIP(hipMalloc((void **)&stage, 2 * expected * sizeof(float)));
    hipError_t e = hipMemcpyAsync(stage, keys, expected * sizeof(float), hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = hipMemcpyAsync(stage + expected, values, expected * sizeof(float), hipMemcpyHostToDevice, s);
    int32_t rc = SKV_OK;
    if (e == hipSuccess) rc = encode_append(L, s, stage, stage + expected, n_rows);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(stage);
    if (e != hipSuccess) return fail_hip(e, "seed: copie hôte→device");
    if (rc) return rc;
    if (e2 != hipSuccess) return fail_hip(e2, "seed: synchronisation");
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_append_host(skv_layer *L, const float *key, const float *value, size_t n_elems) try {
    if (!L || !key || !value) return fail(SKV_ERR_DEVICE, "append: pointeur nul");
    const size_t kv_dim = skv_kv_dim(L);
    if (n_elems != kv_dim)
        return fail(SKV_ERR_DIMENSION, "append KV: attendu " + std::to_string(kv_dim) + ", reçu " +
                                           std::to_string(n_elems));
    if (L->len >= L->capacity)
        return fail(SKV_ERR_DIMENSION,
                    "append KV: capacité " + std::to_string(L->capacity) + " atteinte (overflow)");
    SKV_HIP(hipSetDevice(L->ctx->device));
    hipStream_t s = L->ctx->stream;
    SKV_HIP(hipMemcpyAsync(L->kv_stage, key, kv_dim * sizeof(float), hipMemcpyHostToDevice, s));
    SKV_HIP(hipMemcpyAsync(L->kv_stage + kv_dim, value, kv_dim * sizeof(float), hipMemcpyHostToDevice, s));
    int32_t rc = encode_append(L, s, L->kv_stage, L->kv_stage + kv_dim, 1);
    if (rc) return rc;
    SKV_HIP(hipStreamSynchronize(s));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_append_device(skv_layer *L, skv_stream stream, const void *k_dev, size_t k_off,
                          const void *v_dev, size_t v_off) try {
    if (!L || !k_dev || !v_dev) return fail(SKV_ERR_DEVICE, "append device: pointeur nul");
    if ((k_off | v_off) & 3) return fail(SKV_ERR_DIMENSION, "append device: offset non aligné f32");
    return encode_append(L, as_stream(stream),
                         reinterpret_cast<const float *>((const char *)k_dev + k_off),
                         reinterpret_cast<const float *>((const char *)v_dev + v_off), 1);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_append_batch_device(skv_layer *L, skv_stream stream, const void *k_dev,
                                const void *v_dev, size_t n_rows) try {
    if (!L || !k_dev || !v_dev) return fail(SKV_ERR_DEVICE, "append batch: pointeur nul");
    if (n_rows == 0) return fail(SKV_ERR_DIMENSION, "cache KV batch attend seq > 0");
    return encode_append(L, as_stream(stream), (const float *)k_dev, (const float *)v_dev, n_rows);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_attention_device(skv_layer *L, skv_stream stream, const float *q_dev, float *out_dev,
                             size_t window_start) try {
    if (!L || !q_dev || !out_dev) return fail(SKV_ERR_DEVICE, "attention device: pointeur nul");
    return encode_attention(L, as_stream(stream), q_dev, out_dev, window_start);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_attention_host(skv_layer *L, const float *q, size_t n_elems, size_t window_start,
                           float *out) try {
    if (!L || !q || !out) return fail(SKV_ERR_DEVICE, "attention: pointeur nul");
    if (L->len == 0) return fail(SKV_ERR_DIMENSION, "attention_decode sur KV vide");
    const size_t q_dim = (size_t)L->g.q_heads * L->g.head_dim;
    if (n_elems != q_dim)
        return fail(SKV_ERR_DIMENSION, "attention_decode: q attendu [" + std::to_string(q_dim) +
                                           "], reçu " + std::to_string(n_elems));
    SKV_HIP(hipSetDevice(L->ctx->device));
    hipStream_t s = L->ctx->stream;
    SKV_HIP(hipMemcpyAsync(L->q_stage, q, q_dim * sizeof(float), hipMemcpyHostToDevice, s));
    int32_t rc = encode_attention(L, s, L->q_stage, L->out_stage, window_start);
    if (rc) return rc;
    SKV_HIP(hipMemcpyAsync(out, L->out_stage, q_dim * sizeof(float), hipMemcpyDeviceToHost, s));
    SKV_HIP(hipStreamSynchronize(s));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_decode_step_device(skv_layer *L, skv_stream stream, const void *k_dev, size_t k_off,
                               const void *v_dev, size_t v_off, const float *q_dev,
                               float *out_dev) try {
    if (!L || !k_dev || !v_dev || !q_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "decode_step: pointeur nul");
    const bool fused = tuning().fused_append;
    if (!fused || !uses_flash(L) || !fused_append_built(L)) {
        int32_t rc = skv_append_device(L, stream, k_dev, k_off, v_dev, v_off);
        if (rc) return rc;
        const size_t ws = skv_window_start(L->len - 1, L->window);
        return skv_attention_device(L, stream, q_dev, out_dev, ws);
    }
    if ((k_off | v_off) & 3) return fail(SKV_ERR_DIMENSION, "append device: offset non aligné f32");
    if (L->len >= L->capacity)
        return fail(SKV_ERR_DIMENSION, "append KV résident: capacité " +
                                           std::to_string(L->capacity) + " atteinte (overflow)");
    // the attention kernel writes the row itself: advance the bookkeeping first
    const size_t floor_before = L->floor_pos;
    L->len += 1;
    if (L->g.ring_rows > 0 && L->len > (size_t)L->g.ring_rows)
        L->floor_pos = std::max(L->floor_pos, L->len - (size_t)L->g.ring_rows);
    const size_t ws = skv_window_start(L->len - 1, L->window);
    int32_t rc = encode_attention(L, as_stream(stream), q_dev, out_dev, ws,
                                  reinterpret_cast<const float *>((const char *)k_dev + k_off),
                                  reinterpret_cast<const float *>((const char *)v_dev + v_off));
    if (rc) {
        L->len -= 1;
        L->floor_pos = floor_before;
    }
    return rc;
} catch (...) {
    return skv::fail_exception();
}

// skv_decode_step_device with the split partials in the library's static device array
// instead of the layer's own buffers: nothing here allocates or frees.
int32_t skv_decode_step_static_device(skv_layer *L, skv_stream stream, const void *k_dev, size_t k_off,
                                      const void *v_dev, size_t v_off, const float *q_dev,
                                      float *out_dev) try {
    if (!L || !k_dev || !v_dev || !q_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "decode_step_static: pointeur nul");
    if (!uses_flash(L))
        return fail(SKV_ERR_CONFIG, "decode_step_static: le noyau simple (RETI_RUST_FLASH_SDPA=0) alloue son "
                                    "tampon de scores");
    void *part = L->ctx->static_scratch;
    if (!part) return fail(SKV_ERR_DEVICE, "decode_step_static: tampon statique non résolu");
    if ((k_off | v_off) & 3) return fail(SKV_ERR_DIMENSION, "append device: offset non aligné f32");
    const float *k = reinterpret_cast<const float *>((const char *)k_dev + k_off);
    const float *v = reinterpret_cast<const float *>((const char *)v_dev + v_off);
    hipStream_t s = as_stream(stream);
    if (!tuning().fused_append || !fused_append_built(L)) {
        // separate launches (wide f32 heads have no fused append); on a failure after the
        // append the row stays appended, as with skv_decode_step_device
        int32_t rc = encode_append(L, s, k, v, 1);
        if (rc) return rc;
        return encode_attention(L, s, q_dev, out_dev, skv_window_start(L->len - 1, L->window), nullptr,
                                nullptr, 1, 0.0f, nullptr, part);
    }
    if (L->len >= L->capacity)
        return fail(SKV_ERR_DIMENSION, "append KV résident: capacité " +
                                           std::to_string(L->capacity) + " atteinte (overflow)");
    const size_t floor_before = L->floor_pos;
    L->len += 1;
    if (L->g.ring_rows > 0 && L->len > (size_t)L->g.ring_rows)
        L->floor_pos = std::max(L->floor_pos, L->len - (size_t)L->g.ring_rows);
    int32_t rc = encode_attention(L, s, q_dev, out_dev, skv_window_start(L->len - 1, L->window), k, v, 1,
                                  0.0f, nullptr, part);
    if (rc) {
        L->len -= 1;
        L->floor_pos = floor_before;
    }
    return rc;
} catch (...) {
    return skv::fail_exception();
}

// Whether a chunk's context is to lie over its K or V rows (a caller's activations that share a buffer): every row
// then has to be in the cache before the first context is written.
static bool context_over_rows(const skv_layer *L, size_t c, const float *out, const float *k, const float *v) {
    return over_rows(L->g, out, k, c) || over_rows(L->g, out, v, c);
}

// A chunk of c > 1 rows on a ring layer (bf16, or f32 where the f32 chunk kernel serves the head_dim). The
// ring holds little more than the window, so the chunk's own rows overwrite rows its first queries still attend. They are therefore first
// written to pages of the context's scratch; one launch attends the ring's rows and them, in the
// order of positions, each workgroup only the pages its slots' windows touch; then the rows go
// into the ring. (Two launches around the append, over the old rows and over the new ones,
// each over the whole ring and with partials of its own: 93 us for 512 rows of q16/kv8/hd256 on a
// ring of 1056 rows, against 50 us.)
static int32_t ring_chunk(skv_layer *L, hipStream_t s, const float *q, const float *k, const float *v,
                          size_t c, float *out) {
    const Geom &g = L->g;
    const size_t base = L->len;
    // the rows in the ring that the first query attends (it attends the most of them)
    const size_t lo = std::max(L->floor_pos, skv_window_start(base, L->window));
    ChunkPages pages = layer_pages(g, lo, base);
    pages.new_pos0 = (int)base;
    pages.new_first = (int)(base / 16 * 16);
    const size_t n_new = (base + c - 1) / 16 - base / 16 + 1;
    const size_t pool_bytes = n_new * (size_t)g.page_elems * sizeof(uint16_t); // of K and of V

    DecodeArgs a{};
    {
        RowsAhead ahead(L, c); // the queries are the last c rows
        fill_decode_args(L, q, out, L->floor_pos, nullptr, nullptr, c, tuning().prefill_wgs, a);
    }
    // pages a workgroup of one tile row walks: the window and the workgroup's own rows
    const size_t walked = std::min<size_t>((size_t)pages.n_old + n_new, L->window / 16 + 2);
    const TileShape shape = prefill_shape(g, c * (size_t)g.gqa, walked);
    // f32 pages as terms, made by a launch of their own (see encode_attention), or split by each workgroup
    bool made = g.f32 && f32_terms_pay(g, c) && !capturing(s);
    F32Plan plan{};
    const bool halves = g.f32 && f32_halves(g, c * (size_t)g.gqa, walked);
    // a context over the chunk's own rows is written once they are in the ring, one over its queries once all are read: by the merge, so
    // there has to be one
    const bool late = context_over_rows(L, c, out, k, v) || over_queries(g, out, q, c) || reads_again(g, out, q);
    StreamScratch::Lease lease;
    void *scratch = nullptr;
    int32_t rc = SKV_OK;
    StreamScratch::Lease terms_lease;
    if (made) {
        const int entries = (int)((size_t)pages.n_old + n_new);
        const size_t most = terms_scratch(L, s, (size_t)(entries + 1) / 2, 0, terms_lease, &scratch);
        made = most > 0;
        if (made) {
            plan = plan_f32_chunk(g, c, 0, entries, (int)walked, INT32_MAX, most);
            if (late) plan.splits = std::max(plan.splits, 2);
            a.splits = plan.splits;
            a.splits_total = plan.sets();
            made = a.splits_total == 1 || try_partials(L, s, (size_t)a.splits_total, c, a, lease, 0, nullptr, true) == 0;
        }
    }
    if (!made) {
        a.splits = chunk_splits(g, c, (size_t)(g.f32 ? f32_prefill_slots(g.P, halves) : prefill_tile_slots(g.P, shape)), walked);
        if (late) a.splits = std::max(a.splits, 2);
        a.splits_total = a.splits;
        rc = multi_query_partials(L, s, a.splits > 1 ? (size_t)a.splits : 0, c, a, lease, 2 * pool_bytes, &scratch);
        if (rc) return rc;
    }
    if (made) {
        rc = run_f32_chunk(plan, a, pages, scratch, (int)lo, k, v, s, false);
        if (rc) return rc;
    } else {
        AppendArgs w{};
        w.k_src = k;
        w.v_src = v;
        w.k_pool = static_cast<uint16_t *>(scratch);
        w.v_pool = w.k_pool + pool_bytes / sizeof(uint16_t);
        w.first_pos = (long)(base % 16);
        w.n_rows = (int)c;
        w.g = g;
        w.g.ring_rows = 0;
        SKV_HIP(launch_append(w, s));
        pages.k_new = w.k_pool;
        pages.v_new = w.v_pool;
        SKV_HIP(g.f32 ? launch_f32_prefill(a, pages, nullptr, halves, s) : launch_prefill_tiles(a, pages, shape, s));
    }
    if (a.splits_total == 1) return encode_append(L, s, k, v, c);
    if (late) {
        rc = encode_append(L, s, k, v, c);
        if (rc) return rc;
        SKV_HIP(launch_merge_rows(a, s));
        return SKV_OK;
    }
    SKV_HIP(launch_merge_append(a, append_args(L, k, v, c), s)); // (the caller has checked the capacity)
    appended(L, c);
    return SKV_OK;
}

// The same on an f32 ring layer of wider heads, c <= ring_rows, attended in two phases around the append:
// first every query over the rows already in the ring (capped at the last old position), then, once the chunk is appended,
// over the chunk's own rows (from its first position up to each query's own). Both phases
// leave (o, m, l) partials; one merge produces the context. c <= ring_rows.
static int32_t ring_chunk_f32(skv_layer *L, hipStream_t s, const float *q, const float *k, const float *v,
                              size_t c, float *out) {
    const Geom &g = L->g;
    const size_t base = L->len;
    const size_t tiles = (c * (size_t)g.gqa + 15) / 16 * (size_t)g.kv_heads;
    auto splits_for = [&](int n_pages) {
        size_t want = std::max<size_t>(2 * tuning().prefill_wgs / tiles, 1);
        want = std::min<size_t>(want, std::max<size_t>((size_t)n_pages / 8, 1));
        return (int)std::min<size_t>(want, tuning().prefill_max_splits);
    };
    StreamScratch::Lease lease;
    DecodeArgs a1{}, a3{};
    int s1 = 0;
    if (base > 0) { // phase 1, prepared against the ring as it is now
        fill_decode_args(L, q, out, L->floor_pos, nullptr, nullptr, c, tuning().prefill_wgs, a1, true);
        a1.q_pos0 = (int)base;
        a1.limit_cap = (int)base - 1;
        s1 = splits_for(a1.n_pages);
    }
    const int pages_after = (int)std::min<size_t>((base + c + 15) / 16, (size_t)L->n_pages);
    const int s3 = splits_for(pages_after);
    const int total = s1 + s3;
    if (base > 0) {
        a1.splits = s1;
        a1.split_base = 0;
        a1.splits_total = total;
        int32_t rc = multi_query_partials(L, s, (size_t)total, c, a1, lease);
        if (rc) return rc;
        SKV_HIP(launch_f32_split(a1, s));
    }
    int32_t rc = encode_append(L, s, k, v, c);
    if (rc) return rc;
    fill_decode_args(L, q, out, std::max(base, L->floor_pos), nullptr, nullptr, c, tuning().prefill_wgs, a3, true);
    a3.q_pos0 = (int)base;
    a3.splits = s3;
    a3.split_base = s1;
    a3.splits_total = total;
    if (total > 1) {
        rc = multi_query_partials(L, s, (size_t)total, c, a3, lease);
        if (rc) return rc;
    }
    SKV_HIP(launch_f32_split(a3, s));
    if (total > 1) SKV_HIP(launch_merge_rows(a3, s));
    return SKV_OK;
}

int32_t skv_prefill_chunk_device(skv_layer *L, skv_stream stream, const float *q_dev,
                                 const void *k_dev, const void *v_dev, size_t n_rows,
                                 float *out_dev) try {
    if (!L || !q_dev || !k_dev || !v_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "prefill chunk: pointeur nul");
    if (n_rows == 0) return fail(SKV_ERR_DIMENSION, "attention batch cached shapes: seq == 0");
    if (L->len + n_rows > L->capacity)
        return fail(SKV_ERR_DIMENSION, "append KV résident: capacité " +
                                           std::to_string(L->capacity) + " atteinte (overflow)");
    const size_t kv_dim = skv_kv_dim(L), q_dim = (size_t)L->g.q_heads * L->g.head_dim;
    // f32 ring layers of wide heads take the chunk in steps of at most the ring's rows (see ring_chunk_f32).
    const bool two_phase = L->g.f32 && f32_prefill_slots(L->g.P, false) == 0;
    size_t step = std::min<size_t>(n_rows, 4096);
    if (L->g.ring_rows > 0 && two_phase) step = std::min(step, (size_t)L->g.ring_rows);
    const float *q = q_dev, *k = (const float *)k_dev, *v = (const float *)v_dev;
    float *out = out_dev;
    for (size_t done = 0; done < n_rows; done += step) {
        const size_t c = std::min(step, n_rows - done);
        int32_t rc;
        // the first query attends window - 1 rows in front of the chunk: where none of them (no row at
        // all before the ring is full) is overwritten by the chunk's rows, the chunk is appended first
        // like any other
        const size_t ring = (size_t)L->g.ring_rows;
        if (ring > 0 && c > 1 && L->len + c > ring && c + L->window > ring + 1) {
            rc = (two_phase ? ring_chunk_f32 : ring_chunk)(L, as_stream(stream), q, k, v, c, out);
            if (rc) return rc;
            q += c * q_dim;
            k += c * kv_dim;
            v += c * kv_dim;
            out += c * q_dim;
            continue;
        }
        // a few rows over a full bf16 layer (a speculative verify, the rest of a prompt): the multi-query launch
        // appends them itself, as a decode step's does (its last query tile, which sees all of them, stores them)
        if (c > 1 && c <= (size_t)MQ_APPEND_ROWS && ring == 0 && !L->g.f32 && tuning().fused_append &&
            !context_over_rows(L, c, out, k, v) && !takes_tile_kernel(L->g, c, (L->len + c + 15) / 16)) {
            RowsAhead ahead(L, c);
            rc = encode_attention(L, as_stream(stream), q, out, 0, k, v, c);
            if (rc) return rc;
            ahead.written = true;
            q += c * q_dim;
            k += c * kv_dim;
            v += c * kv_dim;
            out += c * q_dim;
            continue;
        }
        // a chunk that the f32 chunk kernel takes: its rows are stored by the launch that splits its pages into terms
        if (c > 1 && ring == 0 && L->g.f32 && tuning().fused_append && f32_terms_pay(L->g, c) &&
            takes_f32_chunk_kernel(L->g, c, (L->len + c + 15) / 16)) {
            RowsAhead ahead(L, c);
            rc = encode_attention(L, as_stream(stream), q, out, 0, k, v, c);
            if (rc) return rc;
            ahead.written = true;
            q += c * q_dim;
            k += c * kv_dim;
            v += c * kv_dim;
            out += c * q_dim;
            continue;
        }
        rc = encode_append(L, as_stream(stream), k, v, c);
        if (rc) return rc;
        const size_t ws_base = L->g.ring_rows > 0 ? L->floor_pos : 0;
        const size_t first_ws = std::max(ws_base, skv_window_start(L->len - c, L->window));
        if (c == 1) {
            rc = encode_attention(L, as_stream(stream), q, out, first_ws);
        } else {
            rc = encode_attention(L, as_stream(stream), q, out, ws_base, nullptr, nullptr, c);
        }
        if (rc) return rc;
        q += c * q_dim;
        k += c * kv_dim;
        v += c * kv_dim;
        out += c * q_dim;
    }
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_prefill_chunk_host(skv_layer *L, const float *q, const float *k, const float *v,
                               size_t n_rows, float *out) try {
    if (!L || !q || !k || !v || !out) return fail(SKV_ERR_DEVICE, "prefill chunk: pointeur nul");
    if (n_rows == 0) return fail(SKV_ERR_DIMENSION, "attention batch cached shapes: seq == 0");
    SKV_HIP(hipSetDevice(L->ctx->device));
    const size_t kv_dim = skv_kv_dim(L), q_dim = (size_t)L->g.q_heads * L->g.head_dim;
    const size_t qb = n_rows * q_dim * sizeof(float), kb = n_rows * kv_dim * sizeof(float);
    char *buf = nullptr;
    SKV_HIP(hipMalloc((void **)&buf, 2 * qb + 2 * kb));
    float *qd = (float *)buf, *od = (float *)(buf + qb), *kd = (float *)(buf + 2 * qb),
          *vd = (float *)(buf + 2 * qb + kb);
    hipStream_t s = L->ctx->stream;
    hipError_t e = hipMemcpyAsync(qd, q, qb, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(kd, k, kb, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(vd, v, kb, hipMemcpyHostToDevice, s);
    int32_t rc = SKV_OK;
    if (e == hipSuccess) rc = skv_prefill_chunk_device(L, s, qd, kd, vd, n_rows, od);
    if (e == hipSuccess && !rc) e = hipMemcpyAsync(out, od, qb, hipMemcpyDeviceToHost, s);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(buf);
    if (e != hipSuccess) return fail_hip(e, "prefill chunk: copie");
    if (rc) return rc;
    if (e2 != hipSuccess) return fail_hip(e2, "prefill chunk: synchronisation");
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

// ---- the step before the cache: per-head RMSNorm + rotation --------------------------

struct skv_rope {
    CtxRef ctx;
    float *table = nullptr; // [max_positions][rope_dims/2][2]
    size_t max_positions = 0;
    size_t rope_dims = 0;
    int style = 0;
};

int32_t skv_rope_rotations_host(size_t position, size_t rope_dims, size_t frequency_dim, float theta,
                                float position_scale, float *cos_sin_out) try {
    if (!cos_sin_out) return fail(SKV_ERR_DEVICE, "rope: pointeur nul");
    if (rope_dims == 0 || rope_dims % 2 != 0)
        return fail(SKV_ERR_DIMENSION, "RoPE: rope_dims=" + std::to_string(rope_dims) + " doit être pair et non nul");
    if (!(theta > 0.0f)) return fail(SKV_ERR_DIMENSION, "RoPE: theta doit être > 0");
    if (frequency_dim == 0) frequency_dim = rope_dims;
    // rope_rotations (src/decoder/attention_ops.rs:848-887), operation for operation in f32
    volatile float scaled_position = (float)position * position_scale;
    for (size_t pair = 0; pair < rope_dims / 2; ++pair) {
        volatile float exponent = (float)(2 * pair) / (float)frequency_dim;
        volatile float denom = powf(theta, exponent);
        volatile float angle = scaled_position / denom;
        cos_sin_out[2 * pair] = cosf(angle);
        cos_sin_out[2 * pair + 1] = sinf(angle);
    }
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_rope_create(skv_ctx *ctx, size_t max_positions, size_t rope_dims, size_t frequency_dim,
                        float theta, float position_scale, int32_t style, skv_rope **out) try {
    if (!ctx || !out) return fail(SKV_ERR_DEVICE, "skv_rope_create: pointeur nul");
    *out = nullptr;
    if (max_positions == 0 || max_positions > ((size_t)1 << 30))
        return fail(SKV_ERR_CONFIG, "RoPE: nombre de positions invalide");
    if (rope_dims > 512) return fail(SKV_ERR_CONFIG, "RoPE: rope_dims > 512 non supporté");
    if (style != 0 && style != 1) return fail(SKV_ERR_CONFIG, "RoPE: style inconnu");
    // one (cos, sin) pair per position and rotated pair, built on the host: keep it to a
    // size a host vector and a device buffer always hold (1 GiB = 2 M positions at 128 dims)
    if (max_positions * rope_dims > ((size_t)1 << 28))
        return fail(SKV_ERR_CONFIG, "RoPE: table de " + std::to_string(max_positions) + " positions x " +
                                        std::to_string(rope_dims) + " dims au-delà de 1 GiB");
    std::vector<float> host(max_positions * rope_dims);
    for (size_t p = 0; p < max_positions; ++p) {
        int32_t rc = skv_rope_rotations_host(p, rope_dims, frequency_dim, theta, position_scale,
                                             host.data() + p * rope_dims);
        if (rc) return rc;
    }
    SKV_HIP(hipSetDevice(ctx->device));
    skv_rope *r = new skv_rope();
    r->ctx = ctx;
    r->max_positions = max_positions;
    r->rope_dims = rope_dims;
    r->style = style;
    hipError_t e = hipMalloc((void **)&r->table, host.size() * sizeof(float));
    if (e == hipSuccess)
        e = hipMemcpy(r->table, host.data(), host.size() * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        if (r->table) (void)hipFree(r->table);
        delete r;
        return fail_hip(e, "RoPE: table des rotations");
    }
    *out = r;
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

void skv_rope_destroy(skv_rope *rope) {
    if (!rope) return;
    (void)hipSetDevice(rope->ctx->device);
    (void)hipDeviceSynchronize();
    if (rope->table) (void)hipFree(rope->table);
    delete rope;
}

static int32_t check_rope(const skv_rope *rope, size_t position, size_t head_dim) {
    if (!rope) return SKV_OK;
    if (rope->rope_dims > head_dim)
        return fail(SKV_ERR_DIMENSION, "RoPE: rope_dims=" + std::to_string(rope->rope_dims) +
                                           " > head_dim=" + std::to_string(head_dim));
    if (position >= rope->max_positions)
        return fail(SKV_ERR_DIMENSION, "RoPE: position " + std::to_string(position) +
                                           " hors de la table (" + std::to_string(rope->max_positions) + ")");
    return SKV_OK;
}

int32_t skv_rms_norm_rope_decode_device(skv_ctx *ctx, skv_stream stream, const skv_rope *rope,
                                        size_t position, const float *x_dev, const float *weight_dev,
                                        size_t heads, size_t head_dim, float eps, float *out_dev) try {
    if (!ctx || !x_dev || !out_dev) return fail(SKV_ERR_DEVICE, "rms_norm_rope: pointeur nul");
    if (heads == 0 || head_dim == 0 || head_dim > 512 || heads > 65535)
        return fail(SKV_ERR_DIMENSION, "RMSNorm/RoPE heads invalide");
    int32_t rc = check_rope(rope, position, head_dim);
    if (rc) return rc;
    NormRopeArgs a{};
    a.x = x_dev;
    a.out = out_dev;
    a.weight = weight_dev;
    a.rope = rope ? rope->table + position * rope->rope_dims : nullptr;
    a.heads = (int)heads;
    a.head_dim = (int)head_dim;
    a.rope_dims = rope ? (int)rope->rope_dims : 0;
    a.rope_style = rope ? rope->style : 0;
    a.eps = eps;
    SKV_HIP(launch_norm_rope(a, as_stream(stream)));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_rms_norm_rope_rows_device(skv_ctx *ctx, skv_stream stream, const skv_rope *rope,
                                      size_t position_offset, const float *x_dev, const float *weight_dev,
                                      size_t n_rows, size_t heads, size_t head_dim, float eps,
                                      float *out_dev) try {
    if (!ctx || !x_dev || !out_dev) return fail(SKV_ERR_DEVICE, "rms_norm_rope: pointeur nul");
    if (heads == 0 || head_dim == 0 || head_dim > 512 || heads > 65535)
        return fail(SKV_ERR_DIMENSION, "RMSNorm/RoPE heads invalide");
    if (n_rows == 0) return SKV_OK;
    int32_t rc = check_rope(rope, position_offset + n_rows - 1, head_dim);
    if (rc) return rc;
    const size_t row_elems = heads * head_dim;
    for (size_t first = 0; first < n_rows; first += 65535) { // grid y limit
        const size_t n = std::min<size_t>(65535, n_rows - first);
        NormRopeArgs a{};
        a.x = x_dev + first * row_elems;
        a.out = out_dev + first * row_elems;
        a.weight = weight_dev;
        a.rope = rope ? rope->table + (position_offset + first) * rope->rope_dims : nullptr;
        a.heads = (int)heads;
        a.head_dim = (int)head_dim;
        a.rope_dims = rope ? (int)rope->rope_dims : 0;
        a.rope_style = rope ? rope->style : 0;
        a.eps = eps;
        a.n_rows = (int)n;
        SKV_HIP(launch_norm_rope(a, as_stream(stream)));
    }
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_rms_norm_rope_decode_host(skv_ctx *ctx, const float *x, const float *weight, size_t heads,
                                      size_t head_dim, size_t rope_dims, size_t frequency_dim,
                                      size_t position, float eps, float theta, float position_scale,
                                      int32_t style, float *out) try {
    if (!ctx || !x || !out) return fail(SKV_ERR_DEVICE, "rms_norm_rope: pointeur nul");
    if (heads == 0 || head_dim == 0 || head_dim > 512 || heads > 65535)
        return fail(SKV_ERR_DIMENSION, "RMSNorm/RoPE heads invalide");
    if (rope_dims == 0 || rope_dims > head_dim || rope_dims % 2 != 0)
        return fail(SKV_ERR_DIMENSION, "RMSNorm/RoPE: rope_dims invalide");
    if (style != 0 && style != 1) return fail(SKV_ERR_CONFIG, "RoPE: style inconnu");
    std::vector<float> cs(rope_dims);
    int32_t rc = skv_rope_rotations_host(position, rope_dims, frequency_dim, theta, position_scale, cs.data());
    if (rc) return rc;
    SKV_HIP(hipSetDevice(ctx->device));
    const size_t n = heads * head_dim;
    float *buf = nullptr;
    SKV_HIP(hipMalloc((void **)&buf, (2 * n + head_dim + rope_dims) * sizeof(float)));
    float *xd = buf, *od = buf + n, *wd = buf + 2 * n, *rd = wd + head_dim;
    hipStream_t s = ctx->stream;
    hipError_t e = hipMemcpyAsync(xd, x, n * sizeof(float), hipMemcpyHostToDevice, s);
    if (e == hipSuccess && weight) e = hipMemcpyAsync(wd, weight, head_dim * sizeof(float), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(rd, cs.data(), rope_dims * sizeof(float), hipMemcpyHostToDevice, s);
    NormRopeArgs a{};
    a.x = xd;
    a.out = od;
    a.weight = weight ? wd : nullptr;
    a.rope = rd;
    a.heads = (int)heads;
    a.head_dim = (int)head_dim;
    a.rope_dims = (int)rope_dims;
    a.rope_style = style;
    a.eps = eps;
    if (e == hipSuccess) e = launch_norm_rope(a, s);
    if (e == hipSuccess) e = hipMemcpyAsync(out, od, n * sizeof(float), hipMemcpyDeviceToHost, s);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(buf);
    if (e != hipSuccess) return fail_hip(e, "rms_norm_rope");
    if (e2 != hipSuccess) return fail_hip(e2, "rms_norm_rope: synchronisation");
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

static int32_t prekv_step(skv_layer *L, skv_stream stream, const skv_rope *rope, size_t position,
                          const float *q, size_t q_head_stride, const float *gate, const float *k,
                          const float *v, const float *q_norm_w, const float *k_norm_w, float eps,
                          float attn_scalar, float *out_dev) {
    if (!std::isfinite(attn_scalar) || attn_scalar <= 0.0f)
        return fail(SKV_ERR_CONFIG, "scalaire d'attention résident invalide: " + std::to_string(attn_scalar));
    int32_t rc = check_rope(rope, position, (size_t)L->g.head_dim);
    if (rc) return rc;
    if (L->len >= L->capacity)
        return fail(SKV_ERR_DIMENSION, "append KV résident: capacité " +
                                           std::to_string(L->capacity) + " atteinte (overflow)");
    hipStream_t s = as_stream(stream);
    const bool fused = tuning().fused_append;
    if (!fused || !uses_flash(L) || wide_f32_heads(L) || L->g.gqa > 16) {
        // the same step as separate launches: norm + rotation of q and k, append, attention, gate
        NormRopeArgs n{};
        n.x = q;
        n.out = L->q_stage;
        n.weight = q_norm_w;
        n.rope = rope ? rope->table + position * rope->rope_dims : nullptr;
        n.heads = L->g.q_heads;
        n.head_dim = L->g.head_dim;
        n.rope_dims = rope ? (int)rope->rope_dims : 0;
        n.rope_style = rope ? rope->style : 0;
        n.eps = eps;
        n.x_head_stride = (int)q_head_stride;
        SKV_HIP(launch_norm_rope(n, s));
        n.x = k;
        n.out = L->kv_stage;
        n.weight = k_norm_w;
        n.heads = L->g.kv_heads;
        n.x_head_stride = 0;
        SKV_HIP(launch_norm_rope(n, s));
        rc = encode_append(L, s, L->kv_stage, v, 1);
        if (rc) return rc;
        // a context over the gate waits aside until all of it is read
        float *const ctx = gate && over_queries(L->g, out_dev, q, 1, q_head_stride) ? L->out_stage : out_dev;
        rc = encode_attention(L, s, L->q_stage, ctx, skv_window_start(L->len - 1, L->window),
                              nullptr, nullptr, 1, attn_scalar);
        if (rc || !gate) return rc;
        GateArgs ga{};
        ga.ctx = ctx;
        ga.gate = gate;
        ga.out = ctx;
        ga.heads = L->g.q_heads;
        ga.head_dim = L->g.head_dim;
        ga.gate_head_stride = q_head_stride ? (int)q_head_stride : L->g.head_dim;
        SKV_HIP(launch_gate(ga, s));
        if (ctx != out_dev) SKV_HIP(launch_copy(out_dev, ctx, (size_t)L->g.q_heads * L->g.head_dim, s));
        return SKV_OK;
    }
    PreKv pre{};
    pre.rope = rope ? rope->table + position * rope->rope_dims : nullptr;
    pre.q_norm_w = q_norm_w;
    pre.k_norm_w = k_norm_w;
    pre.eps = eps;
    pre.rope_dims = rope ? (int)rope->rope_dims : 0;
    pre.rope_style = rope ? rope->style : 0;
    pre.gate = gate;
    pre.q_head_stride = (int)q_head_stride;
    L->len += 1;
    if (L->g.ring_rows > 0 && L->len > (size_t)L->g.ring_rows)
        L->floor_pos = std::max(L->floor_pos, L->len - (size_t)L->g.ring_rows);
    rc = encode_attention(L, s, q, out_dev, skv_window_start(L->len - 1, L->window), k, v, 1,
                          attn_scalar, &pre);
    if (rc) L->len -= 1;
    return rc;
}

int32_t skv_decode_step_prekv_device(skv_layer *L, skv_stream stream, const skv_rope *rope,
                                     size_t position, const void *q_dev, size_t q_off,
                                     const void *k_dev, size_t k_off, const void *v_dev, size_t v_off,
                                     const float *q_norm_w, const float *k_norm_w, float eps,
                                     float attn_scalar, float *out_dev) try {
    if (!L || !q_dev || !k_dev || !v_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "decode_step_prekv: pointeur nul");
    if ((q_off | k_off | v_off) & 3) return fail(SKV_ERR_DIMENSION, "decode_step_prekv: offset non aligné f32");
    return prekv_step(L, stream, rope, position,
                      reinterpret_cast<const float *>((const char *)q_dev + q_off), 0, nullptr,
                      reinterpret_cast<const float *>((const char *)k_dev + k_off),
                      reinterpret_cast<const float *>((const char *)v_dev + v_off), q_norm_w,
                      k_norm_w, eps, attn_scalar, out_dev);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_decode_step_gated_device(skv_layer *L, skv_stream stream, const skv_rope *rope,
                                     size_t position, const void *qg_dev, size_t qg_off,
                                     const void *k_dev, size_t k_off, const void *v_dev, size_t v_off,
                                     const float *q_norm_w, const float *k_norm_w, float eps,
                                     float attn_scalar, float *out_dev) try {
    if (!L || !qg_dev || !k_dev || !v_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "decode_step_gated: pointeur nul");
    if ((qg_off | k_off | v_off) & 3) return fail(SKV_ERR_DIMENSION, "decode_step_gated: offset non aligné f32");
    // split_q_gate (src/decode_resident/kernels.rs:931-946) by addressing: head h holds its
    // head_dim query values at h * 2 * head_dim and its gate values right after them
    const float *qg = reinterpret_cast<const float *>((const char *)qg_dev + qg_off);
    const size_t hd = (size_t)L->g.head_dim;
    return prekv_step(L, stream, rope, position, qg, 2 * hd, qg + hd,
                      reinterpret_cast<const float *>((const char *)k_dev + k_off),
                      reinterpret_cast<const float *>((const char *)v_dev + v_off), q_norm_w,
                      k_norm_w, eps, attn_scalar, out_dev);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_attn_gate_device(skv_ctx *ctx, skv_stream stream, const float *ctx_dev, const float *gate_dev,
                             size_t gate_head_stride, size_t heads, size_t head_dim, float *out_dev) try {
    if (!ctx || !ctx_dev || !gate_dev || !out_dev) return fail(SKV_ERR_DEVICE, "attn_gate: pointeur nul");
    if (heads == 0 || head_dim == 0 || heads * head_dim > ((size_t)1 << 30))
        return fail(SKV_ERR_DIMENSION, "attn_gate: dimensions invalides");
    if (gate_head_stride != 0 && gate_head_stride < head_dim)
        return fail(SKV_ERR_DIMENSION, "attn_gate: pas du gate < head_dim");
    GateArgs ga{};
    ga.ctx = ctx_dev;
    ga.gate = gate_dev;
    ga.out = out_dev;
    ga.heads = (int)heads;
    ga.head_dim = (int)head_dim;
    ga.gate_head_stride = (int)(gate_head_stride ? gate_head_stride : head_dim);
    SKV_HIP(launch_gate(ga, as_stream(stream)));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_decode_step_batch_device(skv_layer *const *seqs, size_t n_seq, skv_stream stream,
                                     const void *const *k_dev, const void *const *v_dev,
                                     const float *const *q_dev, float *const *out_dev) try {
    if (!seqs || !k_dev || !v_dev || !q_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "decode_step_batch: pointeur nul");
    if (n_seq == 0) return fail(SKV_ERR_DIMENSION, "decode_step_batch: aucune séquence");
    for (size_t i = 0; i < n_seq; ++i) {
        const skv_layer *L = seqs[i];
        if (!L || !k_dev[i] || !v_dev[i] || !q_dev[i] || !out_dev[i])
            return fail(SKV_ERR_DEVICE, "decode_step_batch: pointeur nul (séquence " + std::to_string(i) + ")");
        const Geom &g = L->g, &g0 = seqs[0]->g;
        if (g.q_heads != g0.q_heads || g.kv_heads != g0.kv_heads || g.head_dim != g0.head_dim ||
            (g.ring_rows > 0) != (g0.ring_rows > 0) || g.f32 != g0.f32 || L->window != seqs[0]->window ||
            L->ctx != seqs[0]->ctx)
            return fail(SKV_ERR_DIMENSION, "decode_step_batch: la séquence " + std::to_string(i) +
                                               " n'a pas la géométrie de la séquence 0");
        for (size_t j = 0; j < i; ++j)
            if (seqs[j] == L)
                return fail(SKV_ERR_DIMENSION, "decode_step_batch: séquence " + std::to_string(i) + " en double");
        // nothing is modified unless every sequence can take its row
        if (L->len >= L->capacity)
            return fail(SKV_ERR_DIMENSION, "append KV résident: capacité " + std::to_string(L->capacity) +
                                               " atteinte (overflow), séquence " + std::to_string(i));
    }
    const bool fused = tuning().fused_append;
    if (!fused || !uses_flash(seqs[0]) || seqs[0]->g.gqa > 16 || n_seq == 1 || !fused_append_built(seqs[0])) {
        for (size_t i = 0; i < n_seq; ++i) {
            int32_t rc = skv_decode_step_device(seqs[i], stream, k_dev[i], 0, v_dev[i], 0, q_dev[i], out_dev[i]);
            if (rc) return rc;
        }
        return SKV_OK;
    }
    for (size_t first = 0; first < n_seq; first += SKV_MAX_BATCH) {
        const size_t n = std::min<size_t>(SKV_MAX_BATCH, n_seq - first);
        // the workgroup budget is shared in proportion to the pages each sequence scans
        size_t pages_total = 0;
        for (size_t i = 0; i < n; ++i) {
            const skv_layer *L = seqs[first + i];
            const size_t rows = L->g.ring_rows > 0 ? std::min<size_t>(L->len + 1, (size_t)L->g.ring_rows)
                                                   : L->len + 1 - skv_window_start(L->len, L->window);
            pages_total += (rows + 15) / 16;
        }
        // Sequences, a bit each, whose context lies over some sequence's queries (but its own, exactly) or rows: see over_queries
        const auto look = [&]() -> uint32_t {
            const Geom &g = seqs[0]->g;
            const size_t q_bytes = (size_t)g.q_heads * g.head_dim * sizeof(float), kv_bytes = (size_t)g.kv_heads * g.head_dim * sizeof(float);
            uintptr_t lo = UINTPTR_MAX, hi = 0; // of all contexts: what lies outside lies under none
            for (size_t i = first; i < first + n; ++i) {
                lo = std::min(lo, reinterpret_cast<uintptr_t>(out_dev[i]));
                hi = std::max(hi, reinterpret_cast<uintptr_t>(out_dev[i]) + q_bytes);
            }
            uint32_t over = 0;
            const auto under = [&](const void *in, size_t bytes, const float *own) {
                const uintptr_t at = reinterpret_cast<uintptr_t>(in);
                if (at >= hi || at + bytes <= lo) return;
                for (size_t i = 0; i < n; ++i)
                    if (out_dev[first + i] != own && overlap(out_dev[first + i], q_bytes, in, bytes)) over |= 1u << i;
            };
            for (size_t j = first; j < first + n; ++j) {
                under(q_dev[j], q_bytes, out_dev[j] == q_dev[j] ? out_dev[j] : nullptr);
                under(k_dev[j], kv_bytes, nullptr);
                under(v_dev[j], kv_bytes, nullptr);
            }
            return over;
        };
        DecodeBatchArgs b{};
        size_t floor_before[SKV_MAX_BATCH];
        for (size_t i = 0; i < n; ++i) {
            skv_layer *L = seqs[first + i];
            // the attention kernel writes the row itself: advance the bookkeeping first
            floor_before[i] = L->floor_pos;
            L->len += 1;
            if (L->g.ring_rows > 0 && L->len > (size_t)L->g.ring_rows)
                L->floor_pos = std::max(L->floor_pos, L->len - (size_t)L->g.ring_rows);
        }
        // All contexts stay whole or none does: the merge of one is a launch for all, and a whole one then only walks longer. Batches of two,
        // each by itself / none, us: q8/kv2/hd64 over 370, 400 rows 7.5/6.3, q16/kv2/hd256 over 150, 400 9.3/8.3, q4/kv1/hd128 over 250, 2000
        // 7.7/6.9; four of q32/kv8/hd128 over 250, one of them over 600 8.5/8.0.
        // (Arguments are filled again only where one had stayed whole. Host time of a call, 16 of q32/kv8/hd128 over 4000 rows, all filled
        // twice / once: 13.2/11.9.)
        const int wgs = (int)n * seqs[0]->g.kv_heads, line = whole_step_pages(seqs[0]->g, wgs);
        uint32_t is_short = 0; // a bit each
        for (size_t i = 0; i < n; ++i) {
            const skv_layer *L = seqs[first + i];
            const bool wrapped = L->g.ring_rows > 0 && L->len > (size_t)L->g.ring_rows;
            if (pages_walked(L, skv_window_start(L->len - 1, L->window), wrapped) <= line) is_short |= 1u << i;
        }
        uint32_t over = is_short ? look() : 0;
        const auto fill = [&](size_t i, bool whole_ok) {
            const skv_layer *L = seqs[first + i];
            const size_t ws = skv_window_start(L->len - 1, L->window);
            const size_t rows = L->g.ring_rows > 0 ? std::min<size_t>(L->len, (size_t)L->g.ring_rows) : L->len - ws;
            const size_t share = std::max<size_t>(decode_target_wgs() * ((rows + 15) / 16) / std::max<size_t>(pages_total, 1),
                                                  (size_t)L->g.kv_heads);
            fill_decode_args(L, q_dev[first + i], out_dev[first + i], ws,
                             reinterpret_cast<const float *>(k_dev[first + i]),
                             reinterpret_cast<const float *>(v_dev[first + i]), 1, share, b.seq[i], false, whole_ok, wgs);
        };
        bool split = false, unsplit = false;
        for (size_t i = 0; i < n; ++i) {
            fill(i, over == 0);
            split = split || b.seq[i].splits > 1;
            unsplit = unsplit || b.seq[i].splits == 1;
        }
        for (size_t i = 0; split && over == 0 && i < n; ++i)
            if (is_short >> i & 1) fill(i, false);
        // an unsplit context over what other workgroups read is written aside (see encode_attention)
        if (unsplit && !is_short) over = look();
        for (size_t i = 0; i < n; ++i)
            if ((over >> i & 1) && b.seq[i].splits == 1) b.seq[i].out = seqs[first + i]->out_stage;
        hipError_t e = launch_decode_batch(b, (int)n, as_stream(stream));
        for (size_t i = 0; e == hipSuccess && i < n; ++i)
            if (b.seq[i].out != out_dev[first + i])
                e = launch_copy(out_dev[first + i], b.seq[i].out, (size_t)seqs[0]->g.q_heads * seqs[0]->g.head_dim, as_stream(stream));
        if (e != hipSuccess) {
            for (size_t i = 0; i < n; ++i) {
                seqs[first + i]->len -= 1;
                seqs[first + i]->floor_pos = floor_before[i];
            }
            return fail_hip(e, "decode_step_batch: lancement");
        }
    }
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_decode_step_layers_device(skv_layer *const *layers, size_t n_layers, skv_stream stream,
                                      const void *const *k_dev, const void *const *v_dev,
                                      const float *const *q_dev, float *const *out_dev) try {
    if (!layers || !k_dev || !v_dev || !q_dev || !out_dev)
        return fail(SKV_ERR_DEVICE, "decode_step_layers: pointeur nul");
    for (size_t i = 0; i < n_layers; ++i) {
        int32_t rc = skv_decode_step_device(layers[i], stream, k_dev[i], 0, v_dev[i], 0, q_dev[i],
                                            out_dev[i]);
        if (rc) return rc;
    }
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

static int32_t check_rows(const skv_layer *L, size_t first, size_t n) {
    if (first + n > L->len)
        return fail(SKV_ERR_DIMENSION, "lecture KV lignes " + std::to_string(first) + ".." +
                                           std::to_string(first + n) + " > len " +
                                           std::to_string(L->len));
    if (L->g.ring_rows > 0 && n > 0 && first < L->floor_pos)
        return fail(SKV_ERR_DIMENSION, "lecture KV: ligne " + std::to_string(first) +
                                           " déjà évincée de l'anneau");
    return SKV_OK;
}

int32_t skv_gather_device(skv_layer *L, skv_stream stream, size_t first, size_t n, void *k_dst,
                          void *v_dst) try {
    if (!L) return fail(SKV_ERR_DEVICE, "gather: pointeur nul");
    int32_t rc = check_rows(L, first, n);
    if (rc) return rc;
    if (n == 0) return SKV_OK;
    GatherArgs a{};
    a.k_pool = L->k_pool;
    a.v_pool = L->v_pool;
    a.table = L->table_dev;
    a.k_dst = (uint16_t *)k_dst;
    a.v_dst = (uint16_t *)v_dst;
    a.first_pos = (long)first;
    a.n_rows = (int)n;
    a.g = L->g;
    SKV_HIP(L->g.f32 ? launch_gather_f32(a, as_stream(stream)) : launch_gather(a, as_stream(stream)));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

// Rows of either storage mode as f32 (bf16 rows widened: exact).
int32_t skv_read_rows_f32(skv_layer *L, size_t first, size_t n, float *k_out, float *v_out) try {
    if (!L) return fail(SKV_ERR_DEVICE, "read_rows: pointeur nul");
    int32_t rc = check_rows(L, first, n);
    if (rc) return rc;
    if (n == 0) return SKV_OK;
    const size_t elems = n * skv_kv_dim(L);
    if (!L->g.f32) {
        std::vector<uint16_t> kb(k_out ? elems : 0), vb(v_out ? elems : 0);
        rc = skv_read_rows(L, first, n, k_out ? kb.data() : nullptr, v_out ? vb.data() : nullptr);
        if (rc) return rc;
        auto widen = [](uint16_t b) {
            const uint32_t u = (uint32_t)b << 16;
            float f;
            std::memcpy(&f, &u, sizeof f);
            return f;
        };
        for (size_t i = 0; i < kb.size(); ++i) k_out[i] = widen(kb[i]);
        for (size_t i = 0; i < vb.size(); ++i) v_out[i] = widen(vb[i]);
        return SKV_OK;
    }
    SKV_HIP(hipSetDevice(L->ctx->device));
    float *tmp = nullptr;
    SKV_HIP(hipMalloc((void **)&tmp, 2 * elems * sizeof(float)));
    hipStream_t s = L->ctx->stream;
    float *kd = tmp, *vd = tmp + elems;
    rc = skv_gather_device(L, s, first, n, k_out ? kd : nullptr, v_out ? vd : nullptr);
    hipError_t e = hipSuccess;
    if (!rc && k_out) e = hipMemcpyAsync(k_out, kd, elems * sizeof(float), hipMemcpyDeviceToHost, s);
    if (!rc && e == hipSuccess && v_out) e = hipMemcpyAsync(v_out, vd, elems * sizeof(float), hipMemcpyDeviceToHost, s);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(tmp);
    if (rc) return rc;
    if (e != hipSuccess) return fail_hip(e, "read_rows: copie device→hôte");
    if (e2 != hipSuccess) return fail_hip(e2, "read_rows: synchronisation");
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_read_rows(skv_layer *L, size_t first, size_t n, uint16_t *k_out, uint16_t *v_out) try {
    if (!L) return fail(SKV_ERR_DEVICE, "read_rows: pointeur nul");
    if (L->g.f32) return fail(SKV_ERR_CONFIG, "read_rows: cache f32, lire avec skv_read_rows_f32");
    int32_t rc = check_rows(L, first, n);
    if (rc) return rc;
    if (n == 0) return SKV_OK;
    SKV_HIP(hipSetDevice(L->ctx->device));
    const size_t bytes = n * skv_kv_dim(L) * sizeof(uint16_t);
    uint16_t *tmp = nullptr;
    SKV_HIP(hipMalloc((void **)&tmp, 2 * bytes));
    hipStream_t s = L->ctx->stream;
    uint16_t *kd = tmp, *vd = tmp + n * skv_kv_dim(L);
    rc = skv_gather_device(L, s, first, n, k_out ? kd : nullptr, v_out ? vd : nullptr);
    hipError_t e = hipSuccess;
    if (!rc && k_out) e = hipMemcpyAsync(k_out, kd, bytes, hipMemcpyDeviceToHost, s);
    if (!rc && e == hipSuccess && v_out) e = hipMemcpyAsync(v_out, vd, bytes, hipMemcpyDeviceToHost, s);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(tmp);
    if (rc) return rc;
    if (e != hipSuccess) return fail_hip(e, "read_rows: copie device→hôte");
    if (e2 != hipSuccess) return fail_hip(e2, "read_rows: synchronisation");
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

// ---- measurement aids ---------------------------------------------------------------------
static int32_t probe_read(skv_layer *L, skv_stream stream, bool store_partials) {
    if (!L) return fail(SKV_ERR_DEVICE, "probe: pointeur nul");
    if (L->len == 0) return fail(SKV_ERR_DIMENSION, "probe: cache vide");
    ProbeArgs a{};
    a.k_pool = L->k_pool;
    a.v_pool = L->v_pool;
    a.table = L->table_dev;
    a.sink = nullptr;
    a.n_pages = (int)std::min<size_t>((L->len + 15) / 16, (size_t)L->n_pages);
    a.splits = (int)std::max<size_t>(std::min<size_t>(decode_target_wgs() / (size_t)L->g.kv_heads, (size_t)a.n_pages), 1);
    a.splits = std::min(a.splits, L->max_splits);
    a.g = L->g;
    if (store_partials) {
        // (o[head_dim] per head of the group, rounded down to whole 16-byte units; m and l are 2 of 258 floats)
        a.part = L->part_o;
        a.part_floats = (L->g.gqa * L->g.head_dim) & ~3;
    }
    SKV_HIP(launch_probe_read(a, as_stream(stream)));
    return SKV_OK;
}

int32_t skv_probe_read_pages_device(skv_layer *L, skv_stream stream) try {
    return probe_read(L, stream, false);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_probe_read_store_pages_device(skv_layer *L, skv_stream stream) try {
    return probe_read(L, stream, true);
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_probe_merge_device(skv_layer *L, skv_stream stream, float *out_dev) try {
    if (!L || !out_dev) return fail(SKV_ERR_DEVICE, "probe: pointeur nul");
    if (L->len == 0) return fail(SKV_ERR_DIMENSION, "probe: cache vide");
    if (!uses_flash(L)) return fail(SKV_ERR_CONFIG, "probe: noyau matriciel seulement");
    DecodeArgs a{};
    fill_decode_args(L, nullptr, out_dev, skv_window_start(L->len - 1, L->window), nullptr, nullptr, 1,
                     decode_target_wgs(), a, false, true);
    if (a.splits > 1) SKV_HIP(launch_merge(a, as_stream(stream)));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

int32_t skv_probe_empty_launch_device(skv_ctx *ctx, skv_stream stream) try {
    if (!ctx) return fail(SKV_ERR_DEVICE, "probe: ctx nul");
    SKV_HIP(launch_probe_empty(as_stream(stream)));
    return SKV_OK;
} catch (...) {
    return skv::fail_exception();
}

} // extern "C"

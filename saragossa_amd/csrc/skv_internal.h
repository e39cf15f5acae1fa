// Internal declarations shared by the host side and the kernel launchers.
#pragma once

#include <atomic>
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <exception>
#include <new>
#include <string>

#include "../../include/saragossa_kv.h"

namespace skv {

// ---- errors -------------------------------------------------------------------
void set_error(const std::string &msg);
int32_t fail(int32_t code, const std::string &msg);
// Called from the catch-all of an entry point: the exception in flight becomes a status code
// and a message (nothing C++ crosses the C boundary; the reference never panics on a
// fallible path either).
inline int32_t fail_exception() {
    try {
        throw;
    } catch (const std::bad_alloc &) {
        return fail(SKV_ERR_DEVICE, "mémoire hôte épuisée");
    } catch (const std::exception &e) {
        return fail(SKV_ERR_DEVICE, std::string("exception: ") + e.what());
    } catch (...) {
        return fail(SKV_ERR_DEVICE, "exception inconnue");
    }
}
int32_t fail_hip(hipError_t e, const char *what);

#define SKV_HIP(expr)                                            \
    do {                                                         \
        hipError_t e__ = (expr);                                 \
        if (e__ != hipSuccess) return ::skv::fail_hip(e__, #expr); \
    } while (0)

// ---- geometry of one layer's pages ---------------------------------------------
//
// A page holds 16 rows of K (or V) for every kv head. Inside a page the elements
// are stored in the order the gfx950 matrix instructions read them, so that a
// wavefront fetches one (page, kv head) tile with 16-byte loads from consecutive
// addresses:
//
//   K tile [P/8 groups][16 rows][8 dims]            element (row r, dim d) at
//          ((d/8)*16 + r)*8 + d%8
//   V tile [P/32][4 row-quads][16 cols][2][4 rows]  element (row r, dim d) at
//          ((((d/32)*4 + r/4)*16 + d%16)*2 + (d%32)/16)*4 + r%4
//
// P is head_dim rounded up to 32, 64, 96, 128, 256 or 512; dims in [head_dim, P) stay zero.
struct Geom {
    int q_heads;
    int kv_heads;
    int head_dim;
    int P;          // padded head dim
    int gqa;        // q_heads / kv_heads
    int tile_elems; // one (page, kv head) tile in 16-bit units: P * 16 (bf16), P * 32 (f32)
    int page_elems; // kv_heads * tile_elems
    int ring_rows;  // 0 = full cache; else rows kept by the ring (multiple of 16)
    int f32;        // 1 = the tiles hold f32 (kernels_f32.hip), 0 = bf16
    // slot / gqa as a product: floor(2^(31 + s) / gqa) + 1, s the bits of gqa - 1 (set_gqa)
    uint32_t gqa_mul;
    int gqa_shift;
};
inline void set_gqa(Geom &g) {
    g.gqa = g.q_heads / g.kv_heads;
    g.gqa_shift = 0;
    while ((1l << g.gqa_shift) < g.gqa) ++g.gqa_shift;
    g.gqa_mul = (uint32_t)((1ull << (31 + g.gqa_shift)) / (uint64_t)g.gqa + 1);
}
// Query row of a slot, slot / gqa. Exact below 2^31: the product is too large by at most slot * gqa, less than 2^(31 + s). (A division
// is some thirty instructions, and a chunk's kernel wants five before its first load.)
__host__ __device__ inline int slot_row(const Geom &g, int slot) {
    return (int)((uint32_t)(((uint64_t)((uint32_t)slot * 2) * g.gqa_mul) >> 32) >> g.gqa_shift);
}

// (row, head) of a slot of kv head kvh, counted in heads: where its query and its context lie
__host__ __device__ inline long context_row(const Geom &g, int kvh, int slot) {
    const int row = slot_row(g, slot);
    return (long)row * g.q_heads + kvh * g.gqa + (slot - row * g.gqa);
}

__host__ __device__ inline int k_index(int P, int r, int d) {
    (void)P;
    return (((d >> 3) * 16 + r) << 3) + (d & 7);
}
__host__ __device__ inline int v_index(int P, int r, int d) {
    (void)P;
    return ((((((d >> 5) * 4 + (r >> 2)) * 16 + (d & 15)) * 2 + ((d >> 4) & 1))) << 2) + (r & 3);
}

// The f32 element's tiles (kernels_f32.hip), in floats from the tile's start.
__host__ __device__ inline int k_index_f32(int r, int d) {
    return (((d >> 4) * 64 + ((d >> 2) & 3) * 16 + r) << 2) + (d & 3);
}
__host__ __device__ inline int v_index_f32(int r, int d) {
    return (((d >> 4) * 64 + (r >> 2) * 16 + (d & 15)) << 2) + (r & 3);
}

// Rows are addressed by position; a ring layer keeps position p in slot p % ring_rows.
__host__ __device__ inline long slot_of(long pos, int ring_rows) {
    return ring_rows > 0 ? pos % ring_rows : pos;
}

// ---- launch argument blocks ------------------------------------------------------
struct AppendArgs {
    const float *k_src; // [n_rows, kv_dim] f32
    const float *v_src;
    uint16_t *k_pool;
    uint16_t *v_pool;
    const int32_t *table; // null = page i of the pools is page i of the positions
    long first_pos; // position of the first appended row
    int n_rows;
    int vec;        // K rows may be read 16 bytes at a time (set by the launcher, like what follows)
    int first_page; // logical page of the first row, of a ring the one it has come round to
    int first_row;  // of that page
    int ring_pages; // 0 = not a ring
    Geom g;
};

struct GatherArgs {
    const uint16_t *k_pool;
    const uint16_t *v_pool;
    const int32_t *table;
    uint16_t *k_dst; // [n_rows, kv_dim] bf16 bits
    uint16_t *v_dst;
    long first_pos;
    int n_rows;
    Geom g;
};

// (aligned: in a batch's array no member straddles the scalar unit's 64-byte lines more than in one)
struct alignas(64) DecodeArgs {
    const float *q;  // [n_queries][q_heads*head_dim] f32
    float *out;      // [n_queries][q_heads*head_dim] f32
    const uint16_t *k_pool;
    const uint16_t *v_pool;
    const int32_t *table;
    float *part_o;   // [kv_heads][splits][n_queries*gqa][head_dim]
    float *part_m;   // [kv_heads][splits][n_queries*gqa]   (log2 domain)
    float *part_l;   // [kv_heads][splits][n_queries*gqa]
    int len;          // rows valid: positions 0..len
    int n_queries;    // 1 = decode; C = chunked prefill, query i sits at position q_pos0 + i
    int q_pos0;       // position of query row 0 (len - n_queries unless the chunk is attended in two phases)
    int limit_cap;    // no query attends beyond this position (INT_MAX = only its own causal limit)
    int split_base;   // this launch writes partials [split_base, split_base + splits) of splits_total
    int splits_total; // partial sets the merge will see; 1 = the launch writes the context itself
    int window;       // sliding window applied per query (0 = none)
    int window_start; // first position attended (lower bound for every query)
    int ring_base;    // ring layers: (len-1) - (len-1) % ring_rows
    int ring_t;       // ring layers: (len-1) % ring_rows
    int page_first;   // first logical page scanned
    int n_pages;      // logical pages scanned
    int splits;
    int waves;        // wavefronts per workgroup: 4 or 8
    float qscale;     // (1/sqrt(head_dim)) * log2(e)
    // fused append of the row at position len-1 (k_new null = none)
    const float *k_new; // [kv_dim] f32
    const float *v_new;
    int new_slot;     // slot that receives the row
    int new_page;     // physical page of that slot (the host knows its block table)
    // fused pre-KV step (pre != 0): q and the appended k row arrive raw and get the per-head
    // RMSNorm (weights null = none) and the rotation of this position before they are used
    int pre;
    int rope_dims;          // rotated leading dims of each head (even, <= head_dim; 0 = none)
    int rope_style;         // 0 = halves (i, i + rope_dims/2), 1 = interleaved (2i, 2i+1)
    float eps;
    const float *rope;      // [rope_dims/2][2]: (cos, sin) of this position
    const float *q_norm_w;  // [head_dim]
    const float *k_norm_w;  // [head_dim]
    // decode only: head h of q starts at q + h * q_head_stride (0 = head_dim), and the
    // context of head h is multiplied by sigmoid(gate[h * q_head_stride + col]) (null = none)
    const float *gate;
    int q_head_stride;
    int q_vec;              // q is 16-byte aligned and head_dim a multiple of 8: 16-byte loads
    int xchg_off;           // split kernel: byte offset in LDS of the wavefronts' exchange area (0 = it reuses the staging area); set by the launcher
    Geom g;
};
static_assert(sizeof(DecodeArgs) <= 256, "sixteen of them must fit the kernel argument block");

// The pages a chunk's queries walk, as a list in the order of positions: n_old entries of the
// layer's own pages, then pages outside the layer that hold the chunk's new rows (ring layers,
// whose own pages must not be overwritten while they are still attended; none on full layers).
// Both kinds are aligned to positions that are multiples of 16, so the page in which the new
// rows begin is in the list twice: its old entry speaks for positions below new_pos0, its new one
// for the others.
struct ChunkPages {
    int n_old;           // INT32_MAX = the layer's pages only
    int first_pos;       // position of entry 0's first row
    int start;           // entry e < n_old is table[start + e], less ring_pages when past the ring's end
    int ring_pages;      // 0 = not a ring
    int new_pos0;        // first new position (INT32_MAX = none)
    int new_first;       // position of the first new page's first row
    const uint16_t *k_new; // tiles of the new pages, in order (null: their rows lie in the caller's memory, TermPairs)
    const uint16_t *v_new;
};

// Pages of a chunk's list as three bf16 terms a value (f32 layers): pairs [first, first + held) of entries (2i, 2i + 1), per kv head
// and pair K, then V, three planes each (kernels_f32_prefill.hip).
struct TermPairs {
    void *terms;
    int first, held;
    int entries;        // of the whole list
    int pos_lo, pos_hi; // positions that some query attends
    // the chunk's own rows [kv_dim], from position new_pos to pos_hi: on a full layer to be stored into its pages, on a
    // ring the rows of the list's new entries (new_pos INT32_MAX: all rows are in the layer's pages)
    const float *k_src;
    const float *v_src;
    int new_pos;
    int vec;            // K rows may be read 16 bytes at a time
};

// How a workgroup of the prefill tile kernel divides its work among its wavefronts: one 16-slot
// query tile each; two tiles each (head_dim up to 128); two halves, each half of the
// wavefronts holding the same tiles and walking every other page pair; or four quarters of two
// wavefronts with two tiles each, walking every fourth pair (head_dim 65 to 128).
enum class TileShape { one_tile, two_tiles, halves, quarters };

// Standalone per-head RMSNorm + rotation of one row (the same arithmetic as the fused step).
struct NormRopeArgs {
    const float *x;      // [heads][head_dim]
    float *out;          // [heads][head_dim]
    const float *weight; // [head_dim] or null
    const float *rope;   // [rope_dims/2][2] or null
    int heads, head_dim, rope_dims, rope_style;
    float eps;
    int x_head_stride; // elements between the heads of x (0 = head_dim)
    // several rows at consecutive positions (grid y): row r of x and out is heads * head_dim
    // further (contiguous rows) and uses the rotation of the position r further in the table
    int n_rows;
    unsigned hd4_magic, heads_magic; // wavefront kernel: floor(2^32 / d) + 1 of head_dim / 4 and heads (set by the launcher)
};

// out[h][c] = ctx[h][c] * sigmoid(gate[h * gate_head_stride + c])
struct GateArgs {
    const float *ctx;
    const float *gate;
    float *out;
    int heads, head_dim, gate_head_stride;
};
hipError_t launch_gate(const GateArgs &a, hipStream_t s);
hipError_t launch_copy(float *dst, const float *src, size_t n, hipStream_t s);
hipError_t launch_iota(int32_t *dst, int n, hipStream_t s);

// Measurement aids (a read-only walk of the cache with the decode kernel's pattern; an empty launch).
struct ProbeArgs {
    const uint16_t *k_pool;
    const uint16_t *v_pool;
    const int32_t *table;
    uint32_t *sink;
    float *part;     // null = read only; else every workgroup also writes part_floats floats (a multiple of 4)
    int part_floats;
    int n_pages;
    int splits;
    Geom g;
};
hipError_t launch_probe_read(const ProbeArgs &a, hipStream_t s);
hipError_t launch_probe_empty(hipStream_t s);
hipError_t launch_norm_rope(const NormRopeArgs &a, hipStream_t s);

// Raises a kernel's dynamic LDS limit to the 160 KiB of a gfx950 compute unit, once per
// device and kernel (`done` is a per-kernel bit mask over device ids; the attribute belongs to
// the current device's copy of the code object).
inline hipError_t allow_full_lds(const void *kernel, std::atomic<uint64_t> &done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}

#ifdef __HIPCC__
// max / sum over the four 16-lane rows of a wavefront (lanes l, l^16, l^32, l^48), every
// lane receiving the result: two row swaps in the vector unit instead of two exchanges
// through LDS.
__device__ __forceinline__ float rows_max(float v) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows_sum(float v) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
// Workgroup z of a chunk's grid takes this tile of `per` query slots, the last one first: later rows attend more keys, and where there are
// more workgroups than the device holds at once, or they start one after the other, the short ones then fill what the long ones leave.
// Whole chunks, first tile first / last first, us: multi-query mode, 512 rows of q16/kv8/hd256 over none 21.6/20.0, over 512 30.7/29.8, 256 of
// q32/kv8/hd128 over none 10.8/10.0, 700 of q12/kv4/hd96 over none 14.6/12.8; streaming f32, 384 of q16/kv2/hd256 over 100 49.2/41.6; f32
// by terms, 1024 of q32/kv8/hd128 over none 71.2/61.3. (Not the tile kernel of bf16 layers, whose workgroups fit the device up to 256: 0.7 %
// slower there, 0.3 % faster above.)
__device__ __forceinline__ int longest_first(int n_slots, int per, int z) { return (n_slots - 1) / per - z; }
// sigmoid_scalar (src/decoder/attention_ops.rs:522-524)
__device__ __forceinline__ float sigmoid_gate(float g) { return 1.0f / (1.0f + expf(-g)); }
// The arithmetic of rms_norm_rope_heads_at (src/decoder/attention_ops.rs:682-777), operation
// for operation and without contraction, so that the device row equals the CPU row bit for
// bit when the (cos, sin) table comes from the host's libm.
// (The contraction pragma matters: the __f*_rn intrinsics are plain operators here and
// would be fused into FMAs otherwise.)
__device__ __forceinline__ float head_inv_rms(const float *row, int head_dim, float eps) {
#pragma clang fp contract(off)
    float sum = 0.0f;
    for (int c = 0; c < head_dim; ++c) {
        const float sq = row[c] * row[c];
        sum = sum + sq;
    }
    const float mean_square = sum / (float)head_dim;
    return 1.0f / sqrtf(mean_square + eps);
}
// The same from the squares, already taken (x * x, rounded) and padded with zeros to PADDED entries
// (32, 64, 96 or a multiple of 128) at a 16-byte aligned address: the adds stay in index order, the
// 16-byte loads of a round are asked for before the adds of the round before (asked for four at a time and
// waited for, the LDS's latency was as long again as the adds). LOOP: the loop stays a loop; unrolled, every
// load moves to its top and the page registers of a decode kernel spill.
template <int PADDED, bool LOOP = true>
__device__ __forceinline__ float head_inv_rms_sq(const float *sq, int head_dim, float eps) {
#pragma clang fp contract(off)
    typedef __attribute__((ext_vector_type(4))) float f4;
    constexpr int R = PADDED <= 64 ? PADDED / 8 : PADDED == 96 ? 6 : PADDED <= 128 ? 8 : 4; // units of a round
    constexpr int N = PADDED / (8 * R);                                                     // pairs of rounds
    static_assert(N * 8 * R == PADDED, "every square is added");
    const f4 *p = reinterpret_cast<const f4 *>(sq);
    float sum = 0.0f;
    f4 x[R], y[R];
#pragma unroll
    for (int i = 0; i < R; ++i) x[i] = p[i];
#pragma unroll LOOP ? 1 : N
    for (int k = 0; k < N; ++k) {
#pragma unroll
        for (int i = 0; i < R; ++i) y[i] = p[(2 * k + 1) * R + i];
#pragma unroll
        for (int i = 0; i < R; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = sum + x[i][e];
        }
        const f4 *next = p + (k + 1 < N ? 2 * (k + 1) * R : 0); // (the last round reads a unit it ignores)
#pragma unroll
        for (int i = 0; i < R; ++i) x[i] = next[i];
#pragma unroll
        for (int i = 0; i < R; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = sum + y[i][e];
        }
    }
    const float mean_square = sum / (float)head_dim;
    return 1.0f / sqrtf(mean_square + eps);
}
// Element c of the head after norm (inv, w; w null = 1) and rotation (rope null = none).
__device__ __forceinline__ float norm_rope_elem(const float *row, int c, float inv, const float *w,
                                                const float *rope, int rope_dims, int style) {
#pragma clang fp contract(off)
    auto normed = [&](int i) {
#pragma clang fp contract(off)
        const float scaled = row[i] * inv;
        return w ? scaled * w[i] : scaled;
    };
    if (!rope || c >= rope_dims) return normed(c);
    const int pairs = rope_dims >> 1;
    int pair, i0, i1;
    bool is_first;
    if (style == 1) {
        pair = c >> 1;
        i0 = 2 * pair;
        i1 = i0 + 1;
        is_first = (c & 1) == 0;
    } else {
        is_first = c < pairs;
        pair = is_first ? c : c - pairs;
        i0 = pair;
        i1 = pair + pairs;
    }
    const float cs = rope[2 * pair], sn = rope[2 * pair + 1];
    const float first = normed(i0), second = normed(i1);
    const float fc = first * cs, ss = second * sn, fs = first * sn, sc = second * cs;
    return is_first ? fc - ss : fs + sc;
}
// Four dims of a head, x, after norm and rotation. Interleaved pairs (style 1): r0 holds the unit's two
// (cos, sin). Halves: `other` and `ow` are the partner unit and its weights, r0 and r1 the (cos, sin) of the
// pairs, and the unit lies in the first half or not.
__device__ __forceinline__ __attribute__((ext_vector_type(4))) float
norm_rope_unit(__attribute__((ext_vector_type(4))) float x, __attribute__((ext_vector_type(4))) float other,
               __attribute__((ext_vector_type(4))) float w, __attribute__((ext_vector_type(4))) float ow,
               __attribute__((ext_vector_type(4))) float r0, __attribute__((ext_vector_type(4))) float r1, float inv,
               int style, bool is_first) {
#pragma clang fp contract(off)
    typedef __attribute__((ext_vector_type(4))) float f4;
    f4 n = x * inv;
    n = n * w;
    if (style == 1) {
        const float a0 = n[0] * r0[0], b0 = n[1] * r0[1], c0 = n[0] * r0[1], d0 = n[1] * r0[0];
        const float a1 = n[2] * r0[2], b1 = n[3] * r0[3], c1 = n[2] * r0[3], d1 = n[3] * r0[2];
        return f4{a0 - b0, c0 + d0, a1 - b1, c1 + d1};
    }
    f4 o = other * inv;
    o = o * ow;
    const float cs[4] = {r0[0], r0[2], r1[0], r1[2]};
    const float sn[4] = {r0[1], r0[3], r1[1], r1[3]};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float nc = n[e] * cs[e], os = o[e] * sn[e];
        n[e] = is_first ? nc - os : os + nc;
    }
    return n;
}
#endif

// Rows of a chunk that the decode kernel's multi-query mode can append itself.
constexpr int MQ_APPEND_ROWS = 16;

// One decode step of the same model layer for several independent sequences.
constexpr int SKV_MAX_BATCH = 16;
struct DecodeBatchArgs {
    DecodeArgs seq[SKV_MAX_BATCH];
};
static_assert(sizeof(DecodeBatchArgs) <= 4096, "kernel arguments are limited to 4 KiB");

struct NaiveArgs {
    const float *q;
    float *out;
    const uint16_t *k_pool;
    const uint16_t *v_pool;
    const int32_t *table;
    float *scores; // [q_heads][n_keys]
    long len;
    long window_start;
    float inv_scale; // 1/sqrt(head_dim)
    Geom g;
};

// ---- launchers (kernels.hip) ------------------------------------------------------
hipError_t launch_append(const AppendArgs &a, hipStream_t s);
hipError_t launch_gather(const GatherArgs &a, hipStream_t s);
// f32 storage mode: rows in and out (k_dst / v_dst of GatherArgs then point at f32 rows), and
// the split launch for one query row or a chunk (the caller merges as for bf16)
hipError_t launch_gather_f32(const GatherArgs &a, hipStream_t s);
hipError_t launch_f32_split(const DecodeArgs &a, hipStream_t s);
bool f32_decode_kernel_serves(const DecodeArgs &a); // the launch takes the kernel that can also append the row
hipError_t launch_decode(const DecodeArgs &a, hipStream_t s);
hipError_t launch_decode_batch(const DecodeBatchArgs &b, int n_seq, hipStream_t s);
hipError_t launch_f32_split_batch(const DecodeBatchArgs &b, int n_seq, int max_splits, hipStream_t s);
hipError_t launch_merge(const DecodeArgs &a, hipStream_t s);        // split-K partials -> context
hipError_t launch_prefill_tiles(const DecodeArgs &a, const ChunkPages &c, TileShape shape, hipStream_t s); // chunked prefill, no merge
int prefill_tile_slots(int P, TileShape shape);
hipError_t launch_f32_terms(const DecodeArgs &a, const ChunkPages &c, const TermPairs &t, hipStream_t s); // f32 pages -> terms
size_t f32_terms_bytes(const Geom &g); // of one pair of pages, all kv heads
hipError_t launch_f32_prefill(const DecodeArgs &a, const ChunkPages &c, const TermPairs *t, bool halves, hipStream_t s); // chunked prefill over them (null: over the f32 pages)
int f32_prefill_slots(int P, bool halves); // query slots of a workgroup, 0 = head_dim not served
hipError_t launch_merge_rows(const DecodeArgs &a, hipStream_t s);    // the same merge for many query slots
hipError_t launch_merge_append(const DecodeArgs &a, const AppendArgs &w, hipStream_t s); // that and an append nobody waits for in it
hipError_t launch_naive(const NaiveArgs &a, hipStream_t s);
int decode_max_splits();

} // namespace skv

// gfx950 kernels of the KV hot path, part 5: chunked prefill over the f32 cache on the bf16 matrix
// instruction, with every f32 factor as three bf16 terms.
#include <type_traits>

#include "chunk_pages.h"
#include "f32_terms.h"
#include "lds_copy.h"

namespace skv {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float float4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u4;

namespace {

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// LDS buffers of a group's K or V
__host__ __device__ constexpr int f32_prefill_buffers(int P, bool made) { return made && P <= 128 ? 3 : 2; }
// whether the halves of a workgroup, which hold the same query tiles, make their operands together
__host__ __device__ constexpr bool f32_together(int P, int halves) { return halves > 1 && P > 32; }
// units of those operands, and whether they have LDS of their own; else they lie in the last of three buffers until it is needed
__host__ __device__ constexpr int f32_query_units(int P, int tiles, int waves, int halves) {
    return f32_together(P, halves) ? waves / halves * tiles * (P / 32) * 3 * 64 : 0;
}
__host__ __device__ constexpr bool f32_queries_apart(int P, int tiles, int waves, int halves, bool made) {
    return f32_prefill_buffers(P, made) * halves * 3 * 4 * P + f32_query_units(P, tiles, waves, halves) <= 10240;
}
// steps of `n` done before beat b, spread over the beats [from, to)
__host__ __device__ constexpr int done_before(int b, int n, int from, int to) { return b <= from ? 0 : b >= to ? n : (b - from) * n / (to - from); }

} // namespace

// ------------------------------------------------------------------------------------
// The pages that a chunk attends, split into three bf16 terms, as the operands of f32_prefill_kernel: for every
// kv head and pair of entries of the page list (2i, 2i + 1), K and V, three planes of 4 P units of 16 bytes. K: of both pages one after
// the other, eight dims of a row a unit; V: four keys of a dim from both pages side by side. Keys that nobody attends (before
// the first query's window, past the last row, not the entry's to speak for) are zero in V: zero
// probability times what such a row holds may be NaN (the reference never reads those rows,
// src/decode_resident/kernels.rs:11-88).
// The chunk's own rows are taken from the caller's rows, and on a full layer stored into its pages on the way: the
// append costs no launch of its own (512 rows of q32/kv8/hd128: 4 us).
// Bound by memory: 4 bytes in, 6 out per value (and 4 for a new row's).
// ------------------------------------------------------------------------------------
template <int P, bool RING>
__global__ __launch_bounds__(256) void f32_terms_kernel(DecodeArgs a, ChunkPages c, TermPairs t) {
    constexpr int PLANE = 4 * P;
    constexpr int PARTS = (PLANE + 255) / 256; // workgroups of a pair's K, and of its V: one unit a thread
    const int pair = t.first + (int)blockIdx.x, kvh = blockIdx.y;
    const bool v = blockIdx.z >= PARTS;
    const int tid = (int)threadIdx.x + ((int)blockIdx.z - (v ? PARTS : 0)) * 256;
    const int hd = a.g.head_dim;
    const long kv_dim = (long)a.g.kv_heads * hd;
    u4 *out = reinterpret_cast<u4 *>(t.terms) + (((size_t)kvh * t.held + blockIdx.x) * 2 + (v ? 1 : 0)) * 3 * PLANE;
    // (both entries' places are asked for at once)
    uint32_t place[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) place[h] = entry_place<RING>(a, c, min(2 * pair + h, t.entries - 1));
    const float *tile[2]; // of the pool (an entry of a ring's new rows has none: some tile, not looked at)
    int lo[2], hi[2], pos[2];
    bool own[2]; // every row is the caller's
    // rows of the entry that are the caller's: none, some, all. The first and the last, nearly every page of a chunk, have paths of their
    // own: a test per row made V's loads and stores of 4 bytes each behind a branch (512 rows of q32/kv8/hd128 over 512, this launch
    // 9.5 us -> 8.9; whole chunks over none, 512 29.9 -> 29.3, 50.4 -> 49.6, of q12/kv4/hd96 over 1003 40.1 -> 38.5).
    enum { NONE, SOME, ALL };
    int fresh[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e = min(2 * pair + h, t.entries - 1); // (past the end: the last page again, all of it left out of V)
        own[h] = RING && e >= c.n_old;
        tile[h] = reinterpret_cast<const float *>(v ? a.v_pool : a.k_pool) + (own[h] ? 0 : (size_t)place_tile(a, place[h], kvh) * 4);
        pos[h] = entry_pos<RING>(c, e);
        lo[h] = max(t.pos_lo, entry_lo<RING>(c, e));
        hi[h] = 2 * pair + h < t.entries ? min(t.pos_hi, entry_hi<RING>(c, e)) : -1;
        fresh[h] = own[h] || (!RING && pos[h] >= t.new_pos && pos[h] + 15 <= t.pos_hi) ? ALL : !RING && pos[h] + 15 >= t.new_pos ? SOME : NONE;
    }
    // the caller's row at a position (of an entry that is all the caller's, the nearest one there is)
    const float *rows = (v ? t.v_src : t.k_src) + (long)kvh * hd;
    auto is_new = [&](int h, int p) { return own[h] || (!RING && p >= t.new_pos && p <= t.pos_hi); };
    auto row_at = [&](int p) { return rows + (long)(min(max(p, t.new_pos), t.pos_hi) - t.new_pos) * kv_dim; };
    float4_t x[2];
    {
        const int i = min(tid, PLANE - 1);
        if (v) {
            // four keys of dim d, of either page
            const int d = min((i >> 6) * 16 + (i & 15), hd - 1), key = ((i >> 4) & 3) * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (fresh[h] == NONE) { // uniform
                    x[h] = *reinterpret_cast<const float4_t *>(tile[h] + i * 4);
                } else if (fresh[h] == ALL) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[h][r] = row_at(pos[h] + key + r)[d];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int p = pos[h] + key + r;
                        x[h][r] = *(is_new(h, p) ? row_at(p) + d : tile[h] + i * 4 + r);
                    }
                }
            }
        } else {
            // dims d0 .. d0 + 7 of a row: two units of its tile, 16 apart
            static_assert(PLANE / 2 % 64 == 0, "a wavefront's units are of one page");
            const int pg = __builtin_amdgcn_readfirstlane(i / (PLANE / 2)), du = i - pg * (PLANE / 2), d0 = (du >> 4) * 8;
            const float *k = (pg ? tile[1] : tile[0]) + ((du >> 5) * 64 + ((du >> 4) & 1) * 32 + (du & 15)) * 4;
            const int p = (pg ? pos[1] : pos[0]) + (du & 15);
            const int kind = pg ? fresh[1] : fresh[0];
            const bool nw = kind == ALL || (kind == SOME && is_new(pg, p));
            if (kind == NONE) { // uniform
                x[0] = *reinterpret_cast<const float4_t *>(k);
                x[1] = *reinterpret_cast<const float4_t *>(k + 64);
            } else if (kind == ALL && t.vec) {
                x[0] = *reinterpret_cast<const float4_t *>(row_at(p) + min(d0, hd - 4));
                x[1] = *reinterpret_cast<const float4_t *>(row_at(p) + min(d0 + 4, hd - 4));
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e >> 2][e & 3] = *(nw ? row_at(p) + min(d0 + e, hd - 1) : k + (e >> 2) * 64 + (e & 3));
            }
            if (nw) { // (dims past head_dim hold zero)
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e >> 2][e & 3] = d0 + e < hd ? x[e >> 2][e & 3] : 0.0f;
                if (!RING && (PLANE % 256 == 0 || tid < PLANE)) {
                    float *dst = const_cast<float *>(k);
                    if (d0 < hd) *reinterpret_cast<float4_t *>(dst) = x[0];
                    if (d0 + 4 < hd) *reinterpret_cast<float4_t *>(dst + 64) = x[1];
                }
            }
        }
    }
    {
        const int i = tid;
        if (PLANE % 256 != 0 && i >= PLANE) return;
        if (v) {
            const int d = (i >> 6) * 16 + (i & 15), key = ((i >> 4) & 3) * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (fresh[h] == ALL) {
                    if (d >= hd) x[h] = float4_t{0.f, 0.f, 0.f, 0.f};
                    // (an entry past the end stands for the last page, which its other half stores)
                    else if (!RING && hi[h] >= 0) *reinterpret_cast<float4_t *>(const_cast<float *>(tile[h]) + i * 4) = x[h];
                } else if (fresh[h] == SOME) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const bool nw = is_new(h, pos[h] + key + r);
                        if (nw) x[h][r] = d < hd ? x[h][r] : 0.0f;
                        if (!RING && nw && d < hd && hi[h] >= 0) const_cast<float *>(tile[h])[i * 4 + r] = x[h][r];
                    }
                }
                if (pos[h] >= lo[h] && pos[h] + 15 <= hi[h]) continue; // uniform
#pragma unroll
                for (int r = 0; r < 4; ++r) x[h][r] = pos[h] + key + r >= lo[h] && pos[h] + key + r <= hi[h] ? x[h][r] : 0.0f;
            }
        }
        u4 w[3];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t t0, t1, t2;
            three_terms(x[k >> 1][(k & 1) * 2], x[k >> 1][(k & 1) * 2 + 1], t0, t1, t2);
            w[0][k] = t0;
            w[1][k] = t1;
            w[2][k] = t2;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) out[k * PLANE + i] = w[k];
    }
}

// ------------------------------------------------------------------------------------
// prefill_tile_kernel (kernels_prefill.hip) on f32 pages: the same slots, splits, page list, softmax
// base and pipeline (scores of the next group with this group's exponentials between them, then this
// group's accumulation). Six bf16 products of three-term factors replace one f32 product: the f32
// instruction does 4 keys' or dims' worth in the cycles in which the bf16 one does 64, so six
// are 2.6 times as fast (157 TFLOP/s against 2.5 PFLOP/s / 6), and no less exact: the factors are
// split without a rounding, what is left out is at most 2^-24 of a product (f32_terms.h), and sums are
// in f32 in both.
//
// MADE: the pages come as terms from f32_terms_kernel's scratch, straight to LDS: K of a group of pairs, V of the group before
// it, K of the next group and so on, an item each, in three buffers in turn (two at head_dim 256). A barrier stands behind
// each item; the copies of an item are issued two items ahead (one at 256). Otherwise pages come through registers, where all
// threads split each value once for the whole workgroup, and go to LDS as three planes of bf16 operands. K and V have one
// buffer each: V of a group of pairs is stored while the scores of the next group are computed, K of the group after
// that while the accumulation runs, with a barrier behind each window; the loads are issued a window ahead.
// Bound by the matrix pipes, which run at 1.4 PFLOP/s on long walks. 512 rows as one call on layers that are in no cache, in us on
// one MI355X, split by the workgroup / made: q32/kv8/hd128 over 0, 512, 1024, 4096, 16384 rows 35.0/30.1, 57.8/50.3, 80.1/69.5,
// 187/183, 632/627; q16/kv2/hd256 over 1024, 4096 80.7/75.0, 188/173. (f32_split_kernel, kernels_f32.hip, over 512, 16384 of the
// former 83.5, 1267.) At head_dim 256 the third terms of the queries live in LDS: in registers they spill.
// ------------------------------------------------------------------------------------
template <int P, int TILES, int WAVES, int HALVES, bool RING, bool MADE>
__global__ __launch_bounds__(WAVES * 64) void f32_prefill_kernel(DecodeArgs a, ChunkPages c, TermPairs terms) {
    constexpr int THREADS = WAVES * 64;
    constexpr int KK = P / 32;
    constexpr int NT = P / 16;
    constexpr int PLANE = 4 * P;                 // 16-byte units of one term of a pair's K (or V)
    constexpr int ITEM = HALVES * 3 * PLANE;     // units of a group's K (or V): [half][term][PLANE]
    constexpr int GP = 2 * HALVES;               // pages of a group: a pair for each half
    constexpr int NBUF = f32_prefill_buffers(P, MADE);
    constexpr int HALF_KIB = 3 * PLANE / 64;
    // MADE: KiB of an item that a wavefront copies (of two pairs: a number that divides a pair's)
    constexpr int CPW = [] {
        int n = (ITEM / 64 + WAVES - 1) / WAVES;
        while (HALVES > 1 && HALF_KIB % n != 0) ++n;
        return n;
    }();
    constexpr int CU = (HALVES * PLANE + THREADS - 1) / THREADS; // else: units of K, and of V, a thread makes per group
    constexpr bool FULL = HALVES * PLANE % THREADS == 0;
    constexpr bool TOGETHER = f32_together(P, HALVES);
    static_assert(!TOGETHER || P <= 128, "all three terms are in registers");
    constexpr bool Q_APART = f32_queries_apart(P, TILES, WAVES, HALVES, MADE);
    constexpr int Q_AT = Q_APART ? NBUF * ITEM : 2 * ITEM;
    static_assert(Q_APART || (NBUF == 3 && f32_query_units(P, TILES, WAVES, HALVES) <= ITEM), "the queries fit the buffer that is free");
    extern __shared__ __attribute__((aligned(16))) u4 kv_planes[]; // [NBUF][ITEM] (not MADE: K, V)
    constexpr int V_AT = ITEM;

    const Geom g = a.g;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int j = lane >> 4;
    const int split = blockIdx.x;
    const int kvh = blockIdx.y;
    const int G = g.gqa;
    const int n_slots = a.n_queries * G;
    constexpr int TW = WAVES / HALVES;
    const int half = HALVES > 1 ? wave / TW : 0;
    const int tw = HALVES > 1 ? wave % TW : wave;
    const int wg_slot0 = longest_first(n_slots, TW * TILES * 16, blockIdx.z) * (TW * TILES * 16);
    const int wg_slot1 = min(n_slots, wg_slot0 + TW * TILES * 16) - 1;

    auto limit_of = [&](int slot) { return a.q_pos0 + slot_row(a.g, slot); };
    auto ws_of = [&](int slot) { return a.window > 0 ? max(a.window_start, limit_of(slot) + 1 - a.window) : a.window_start; };
    const int wg_ws_lo = ws_of(wg_slot0);
    const int wg_lim_hi = limit_of(wg_slot1);
    auto entry_of = [&](int pos) {
        if (!RING) return pos >> 4;
        return pos < c.new_pos0 ? max((pos - c.first_pos) >> 4, 0) : c.n_old + ((pos - c.new_first) >> 4);
    };
    // Entries [pb0, pb1) of the page list: what any slot of the workgroup can see, divided among the splits; of made terms whole
    // pairs (2i, 2i + 1) of those at hand.
    const int e_lo = entry_of(wg_ws_lo);
    const int e_hi = entry_of(wg_lim_hi) + 1;
    const int p_lo = MADE ? max(e_lo >> 1, terms.first) : e_lo;
    const int p_hi = MADE ? max(min((e_hi + 1) >> 1, terms.first + terms.held), p_lo) : e_hi;
    const unsigned span = (unsigned)(p_hi - p_lo);
    const int p0 = p_lo + (int)(((unsigned)split * span) / (unsigned)a.splits);
    const int p1 = p_lo + (int)(((unsigned)(split + 1) * span) / (unsigned)a.splits);
    const int pb0 = MADE ? 2 * p0 : p0, pb1 = MADE ? 2 * p1 : p1;
    const int n_it = pb1 - pb0;
    const int n_groups = (n_it + GP - 1) / GP;

    // ---- MADE: copies, memory -> LDS. Item 0 is K of the first group, then V of group g is item 2 g + 2 and K of group g + 1
    // item 2 g + 1. Pairs past the end are the last one again, unused.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)kv_planes;
    const uint32_t lane_at = (uint32_t)lane * 16;
    static_assert(!MADE || HALF_KIB % CPW == 0 || HALVES == 1, "a wavefront copies from one pair");
    const int kib0 = min(wave * CPW, ITEM / 64 - CPW); // (the last ones may copy the same)
    const u4 *const terms_kvh = reinterpret_cast<const u4 *>(terms.terms) + (size_t)kvh * terms.held * 2 * 3 * PLANE;
    struct Item {
        const u4 *from;
        uint32_t lds;
    };
    auto item_of = [&](int group, bool v, int buf) __attribute__((always_inline)) {
        const int h = HALVES > 1 ? kib0 / HALF_KIB : 0;
        const int pr = max(min(p0 + group * HALVES + h, terms.first + terms.held - 1) - terms.first, 0);
        Item it;
        it.from = terms_kvh + ((size_t)(pr * 2 + (v ? 1 : 0)) * HALF_KIB + (kib0 - h * HALF_KIB)) * 64;
        it.lds = lds0 + (uint32_t)(buf * ITEM + kib0 * 64) * 16;
        return it;
    };
    auto copy_kib = [&](const Item &it, int k) __attribute__((always_inline)) {
        copy_to_lds(it.from + (k >> 2) * 256, lane_at, it.lds + (uint32_t)(k >> 2) * 4096, k & 3);
    };
    // (past the end: a page again, unused; of made terms nothing is fetched by entry)
    auto entry = [&](int it) { return MADE ? pb0 + it : min(pb0 + it, e_hi - 1); };

    // ---- not MADE: pages, memory -> registers, where all threads split each value once for the whole workgroup, then LDS. Places of the tiles one per lane, asked for a group ahead and
    // read with v_readlane (a scalar read of the table would stall every LDS read in flight).
    uint32_t ids;
    auto ask_ids = [&](int it) __attribute__((always_inline)) { ids = entry_tile<RING>(a, c, entry(it + lane), kvh); };
    auto tile_of = [&](int it0, int d, bool v) __attribute__((always_inline)) {
        const uint16_t *pool = v ? a.v_pool : a.k_pool;
        if (RING && entry(it0 + d) >= c.n_old) pool = v ? c.v_new : c.k_new;
        return reinterpret_cast<const float4_t *>(pool) + (uint32_t)__builtin_amdgcn_readlane(ids, d);
    };
    // unit u of a thread, of the PLANE * HALVES bf16 units of a group: eight dims of a row of K (two
    // f32 units 16 apart), or four keys of a dim from both pages of V
    // At head_dim 256 K and V take turns in the same registers: loads go out at the end of a window and
    // are split in the second half of the next.
    constexpr bool SHARE = !MADE && P > 128;
    float4_t kx[CU][2], vx_own[SHARE ? 1 : CU][2];
    float4_t(&vx)[CU][2] = [&]() -> float4_t(&)[CU][2] {
        if constexpr (SHARE) return kx;
        else return vx_own;
    }();
    // (places as unsigned numbers: the remainder by a power of two of a signed one, which the compiler does not know to be positive, takes
    // registers that head_dim 256 does not have: a ring chunk of 64 rows of q16/kv8/hd256 67.0 us against 62.2)
    auto load_k = [&](int it0, int d) __attribute__((always_inline)) { // pages it0 + d ..
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            const int i = tid + u * THREADS;
            const int pg = min(__builtin_amdgcn_readfirstlane(i / (PLANE / 2)), GP - 1);
            const int du = (int)((unsigned)i % (PLANE / 2));
            const float4_t *t = tile_of(it0, d + pg, false) + (du >> 5) * 64 + ((du >> 4) & 1) * 32 + (du & 15);
            kx[u][0] = t[0];
            kx[u][1] = t[16];
        }
    };
    auto load_v = [&](int it0, int d) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            const int i = tid + u * THREADS;
            const int pr = min(__builtin_amdgcn_readfirstlane(i / PLANE), HALVES - 1);
            vx[u][0] = tile_of(it0, d + 2 * pr, true)[(unsigned)i % PLANE];
            vx[u][1] = tile_of(it0, d + 2 * pr + 1, true)[(unsigned)i % PLANE];
        }
    };
    // Keys that no slot of the workgroup attends: zero probability, but 0 x NaN is NaN, so on the
    // pages at the edges of the attended range their V values become zero in the registers (the
    // reference never reads those rows, src/decode_resident/kernels.rs:11-88).
    const Inner wg_in = inner_entries<RING>(c, pb0, pb1, wg_ws_lo, wg_lim_hi);
    auto mask_v = [&](int first_page) __attribute__((always_inline)) {
        const int e0 = pb0 + first_page, e1 = e0 + GP;
        if ((e0 >= wg_in.o0 && e1 <= wg_in.o1) || (RING && e0 >= wg_in.n0 && e1 <= wg_in.n1)) return; // uniform
#pragma unroll
        for (int u = 0; u < CU; ++u) {
            const int i = tid + u * THREADS;
            const int pr = __builtin_amdgcn_readfirstlane(i / PLANE);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int it = first_page + 2 * pr + h;
                const int e = entry(it);
                const int pos0 = entry_pos<RING>(c, e) + ((i >> 4) & 3) * 4;
                const int lo = max(wg_ws_lo, entry_lo<RING>(c, e)), hi = min(wg_lim_hi, entry_hi<RING>(c, e));
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    vx[u][h][r] = it < n_it && pos0 + r >= lo && pos0 + r <= hi ? vx[u][h][r] : 0.0f;
            }
        }
    };
    // Splitting in small steps that can stand between products: step s splits two values of unit s / 4;
    // the unit's last step stores its three terms.
    constexpr int SPLIT_STEPS = CU * 4;
    uint32_t t0[4], t1[4], t2[4];
    auto split_step = [&](int s, bool v) __attribute__((always_inline)) {
        const int u = s >> 2, k = s & 3;
        const float4_t x = v ? vx[u][k >> 1] : kx[u][k >> 1];
        three_terms((k & 1) ? x[2] : x[0], (k & 1) ? x[3] : x[1], t0[k], t1[k], t2[k]);
        if (k == 3) {
            const int i = tid + u * THREADS;
            // K: [half][term][page of the pair][P/2 * 4 units]; V: [half][term][PLANE]
            const int h = i / PLANE;
            if (FULL || h < HALVES) {
                u4 *dst = kv_planes + (v ? V_AT : 0) + h * 3 * PLANE + (unsigned)i % PLANE;
                dst[0] = u4{t0[0], t0[1], t0[2], t0[3]};
                dst[PLANE] = u4{t1[0], t1[1], t1[2], t1[3]};
                dst[2 * PLANE] = u4{t2[0], t2[1], t2[2], t2[3]};
            }
        }
    };

    if constexpr (!MADE) {
        ask_ids(0);
        load_k(0, 0);
    }
    // ---- this wavefront's query tiles: their loads, the first item's copies, the conversion, further items
    int my_limit[TILES], my_ws[TILES];
    int t_ws_hi[TILES], t_lim_lo[TILES];
    bool t_on[TILES];
    // (at head_dim 256 the third terms, used once per K-step and page, live in LDS behind the planes)
    constexpr int QT = P > 128 ? 2 : 3;
    bf16x8_t q[TILES][KK][QT];
    // Halves load a half of their tiles' K-steps each and find the others' in LDS behind the first barrier (see prefill_tile_kernel; 512 rows
    // of q32/kv8/hd128 over 0, 512 30.9 -> 30.1, 51.7 -> 51.0 us, of q8/kv2/hd64 over 2000 28.4 -> 27.9).
    constexpr int QK = TOGETHER ? (KK + HALVES - 1) / HALVES : KK;
    auto share = [&](int i) { return TOGETHER ? min(half * QK + i, KK - 1) : i; }; // (the last part may make one again)
    u4 *const queries = kv_planes + Q_AT + tw * TILES * KK * 3 * 64 + lane; // of this wavefront's tiles
    float qv[TILES][QK][8];
    u4 *q_third = kv_planes + NBUF * ITEM + wave * TILES * KK * 64 + lane; // the wavefront's own
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int s0 = wg_slot0 + (tw * TILES + t) * 16;
        t_on[t] = s0 < n_slots;
        const int s_last = min(s0 + 15, n_slots - 1);
        const int my_slot = min(s0 + n, n_slots - 1);
        my_limit[t] = limit_of(my_slot);
        my_ws[t] = ws_of(my_slot);
        t_lim_lo[t] = limit_of(min(s0, n_slots - 1));
        t_ws_hi[t] = ws_of(s_last);
        const float *qrow = a.q + context_row(g, kvh, my_slot) * g.head_dim;
        if (a.q_vec) {
#pragma unroll
            for (int kk = 0; kk < QK; ++kk) {
                const float4_t *qp = reinterpret_cast<const float4_t *>(qrow + min(share(kk) * 32 + j * 8, g.head_dim - 8));
                const float4_t x0 = qp[0], x1 = qp[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    qv[t][kk][e] = x0[e];
                    qv[t][kk][4 + e] = x1[e];
                }
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < QK; ++kk) {
#pragma unroll
                for (int e = 0; e < 8; ++e) qv[t][kk][e] = qrow[min(share(kk) * 32 + j * 8 + e, g.head_dim - 1)];
            }
        }
    }
    if constexpr (MADE) {
        const Item first = item_of(0, false, 0);
#pragma unroll
        for (int k = 0; k < CPW; ++k) copy_kib(first, k);
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int kk = 0; kk < QK; ++kk) {
            uint32_t w[3][4];
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) {
                const int d = share(kk) * 32 + j * 8 + e2 * 2;
                const float x = d < g.head_dim ? qv[t][kk][e2 * 2] * a.qscale : 0.0f;
                const float y = d + 1 < g.head_dim ? qv[t][kk][e2 * 2 + 1] * a.qscale : 0.0f;
                three_terms(x, y, w[0][e2], w[1][e2], w[2][e2]);
            }
            if constexpr (TOGETHER) {
#pragma unroll
                for (int k = 0; k < 3; ++k) queries[((t * KK + share(kk)) * 3 + k) * 64] = u4{w[k][0], w[k][1], w[k][2], w[k][3]};
            } else {
#pragma unroll
                for (int k = 0; k < QT; ++k) q[t][kk][k] = __builtin_bit_cast(bf16x8_t, u4{w[k][0], w[k][1], w[k][2], w[k][3]});
            }
            if constexpr (QT == 2) q_third[(t * KK + kk) * 64] = u4{w[2][0], w[2][1], w[2][2], w[2][3]};
        }
    }
    if constexpr (MADE && NBUF == 3) {
        copies_landed(); // (the compiler has waited for the queries, and so for these copies)
        const Item second = item_of(1, false, 1);
#pragma unroll
        for (int k = 0; k < CPW; ++k) copy_kib(second, k);
    }

    // Up to head_dim 128 the leading products and the other five, 2^-8 of them, have sums of their own: an
    // addition cuts off what is far below its sum. Errors against 64 bits, sums apart / together / the kernel of f32
    // products: 512 rows of q32/kv8/hd128 over 1536 3.1e-7/5.3e-7/4.5e-7, over none 2.0e-7/2.4e-7/2.1e-7, of q8/kv2/hd64
    // over 2000 2.1e-7/3.3e-7/3.6e-7. At 256, where there are no registers for it (together / f32 products):
    // q16/kv2 over 4000 6.4e-7/6.8e-7, q16/kv8 on a ring of 1024 4.4e-7/4.0e-7.
    constexpr bool APART = P <= 128;
    float4_t o[TILES][NT], o_low[TILES][APART ? NT : 1];
    // The base of a slot's softmax lags up to 8 behind its largest score, so weights reach 2^8 and the
    // accumulators start close to zero, where their sums are most exact (512 rows of q32/kv8/hd128 over 1536: errors of 5.3e-7 against 64
    // bits, 1.3e-6 with the base 8 ahead). Sums of values near the top of the range that pass
    // through an infinity for it are taken again at the end.
    float4_t neg_m[TILES];
    float m_base[TILES], l_run[TILES];
    // a score whose bits reach thr_i moves its slot's base: SEEN (any above 8), or, for a slot without a key so far, UNSEEN
    // (whatever it is). Where registers are short (head_dim 256, terms not made) scores are compared as floats, with 8 or -inf.
    constexpr bool BITS = MADE || P <= 128;
    constexpr int UNSEEN = BITS ? INT32_MIN : (int)0xff800000, SEEN = BITS ? 0x41000001 : 0x41000000;
    int thr_i[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int u = 0; u < NT; ++u) o[t][u] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < (APART ? NT : 0); ++u) o_low[t][u] = float4_t{0.f, 0.f, 0.f, 0.f};
        m_base[t] = 0.0f;
        neg_m[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        thr_i[t] = UNSEEN;
        l_run[t] = 0.0f;
    }
    float4_t sa[TILES], sb[TILES];
    bf16x8_t p[TILES][3];

    int in0, in1, in2, in3; // pairs whose keys every slot of the wavefront attends
    {
        int lo = t_ws_hi[0], hi = t_lim_lo[0];
#pragma unroll
        for (int t = 1; t < TILES; ++t) {
            lo = max(lo, t_ws_hi[t]);
            hi = min(hi, t_lim_lo[t]);
        }
        const Inner r = inner_entries<RING>(c, pb0, pb1, lo, hi); // (pairs of a range that starts at an even entry)
        in0 = (r.o0 - pb0 + 1) >> 1;
        in1 = (r.o1 - pb0) >> 1;
        in2 = (r.n0 - pb0 + 1) >> 1;
        in3 = (r.n1 - pb0) >> 1;
    }
    // scores of keys outside the slot's range become -inf
    auto mask = [&](int pair) __attribute__((always_inline)) {
        if ((pair >= in0 && pair < in1) || (RING && pair >= in2 && pair < in3)) return; // uniform
        const int it = 2 * pair;
        const int ea = entry(it), eb = entry(it + 1);
        const int pos_a = entry_pos<RING>(c, ea), pos_b = entry_pos<RING>(c, eb);
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const int lo_a = max(my_ws[t], entry_lo<RING>(c, ea)), hi_a = min(my_limit[t], entry_hi<RING>(c, ea));
            const int lo_b = max(my_ws[t], entry_lo<RING>(c, eb)), hi_b = min(my_limit[t], entry_hi<RING>(c, eb));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int pa = pos_a + j * 4 + e, pb = pos_b + j * 4 + e;
                sa[t][e] = it < n_it && pa >= lo_a && pa <= hi_a ? sa[t][e] : -INFINITY;
                sb[t][e] = it + 1 < n_it && pb >= lo_b && pb <= hi_b ? sb[t][e] : -INFINITY;
            }
        }
    };
    // the largest of a lane's scores, as integers of their bits (positive floats in their order, any other below them)
    int mi[TILES];
    auto top_step = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float4_t &x = q < 2 ? sa[t] : sb[t];
            const int m = max(__float_as_int(x[q & 1 ? 2 : 0]), __float_as_int(x[q & 1 ? 3 : 1]));
            mi[t] = q == 0 ? m : max(m, mi[t]);
        }
    };
    // where a score passes the base by more than 8, the wavefront's bases move
    auto settle = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float mx = fmaxf(fmaxf(fmaxf(sa[t][0], sa[t][1]), fmaxf(sa[t][2], sa[t][3])),
                                   fmaxf(fmaxf(sb[t][0], sb[t][1]), fmaxf(sb[t][2], sb[t][3])));
            if (__builtin_amdgcn_ballot_w64(BITS ? mi[t] >= thr_i[t] : mx > __int_as_float(thr_i[t]))) {
                const float top = rows_max(mx);
                const bool unseen = thr_i[t] < 0;
                const float d = unseen ? (top == -INFINITY ? 0.0f : top) : fmaxf(top, 0.0f);
                const float alpha = unseen ? 1.0f : fast_exp2(-d);
                m_base[t] += d;
                neg_m[t] = float4_t{-m_base[t], -m_base[t], -m_base[t], -m_base[t]};
                thr_i[t] = unseen && top == -INFINITY ? UNSEEN : SEEN;
                l_run[t] *= alpha;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sa[t][e] -= d;
                    sb[t][e] -= d;
                }
                if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
                    for (int u = 0; u < NT; ++u) o[t][u] *= alpha;
#pragma unroll
                    for (int u = 0; u < (APART ? NT : 0); ++u) o_low[t][u] *= alpha;
                }
            }
        }
    };

    // probabilities of the settled scores in nine steps: exponential of score s, every other one the
    // three terms of the two before it
    float pe[TILES][2];
    uint32_t pw[TILES][3][4];
    auto prob_step = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (s >= 2 && (s & 1) == 0) {
                l_run[t] += pe[t][0];
                l_run[t] += pe[t][1];
                const int k = (s >> 1) - 1;
                three_terms(pe[t][0], pe[t][1], pw[t][0][k], pw[t][1][k], pw[t][2][k]);
            }
            if (s < 8) pe[t][s & 1] = fast_exp2(s < 4 ? sa[t][s & 3] : sb[t][s & 3]);
        }
    };

    const u4 *const planes = kv_planes + half * 3 * PLANE + lane;
    const u4 *const v_planes = kv_planes + V_AT + half * 3 * PLANE + lane; // not MADE
    constexpr int BEATS = 2 * KK * 6;
    static_assert(BEATS >= 9 && (MADE ? BEATS >= 2 * CPW : BEATS >= SPLIT_STEPS * (SHARE ? 2 : 1)), "at most one step of a kind between two products");
    // operand set `at` of a window, K-step at / 2 of page A or B, dim tile `at` of V: three terms
    u4 op[2 * KK][3];
    u4 q2[KK][TILES]; // QT == 2: the third terms of K-step at / 2
    auto ask_k = [&](const u4 *k_half, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) op[at][k] = k_half[k * PLANE + (at & 1) * (PLANE / 2) + (at >> 1) * 64];
        if constexpr (QT == 2) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                if ((at & 1) == 0) q2[at >> 1][t] = q_third[(t * KK + (at >> 1)) * 64];
        }
    };
    auto ask_v = [&](const u4 *v_half, int at) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) op[at][k] = v_half[k * PLANE + at * 64];
    };
    // What the next window's operands need, between the products of this one, behind beat b: copies of `next` over the first half of
    // the window, or steps of splitting (V where the scores are computed, K two groups on where they are accumulated).
    auto copies = [&](const Item &next, int b) __attribute__((always_inline)) {
        constexpr int EVERY = MADE ? BEATS / 2 / CPW : 1;
        if (b % EVERY == 0 && b / EVERY < CPW) copy_kib(next, b / EVERY);
    };
    auto feed = [&](const Item &next, bool v, int b) __attribute__((always_inline)) {
        if constexpr (MADE) {
            copies(next, b);
        } else {
            constexpr int S_FROM = SHARE ? BEATS / 2 : 0;
            const int ss = done_before(b, SPLIT_STEPS, S_FROM, BEATS);
            if (done_before(b + 1, SPLIT_STEPS, S_FROM, BEATS) > ss) split_step(ss, v);
        }
    };
    // window 1: scores of the next group, between them the probabilities of this one
    auto scores = [&](const u4 *k_half, const Item &next, auto first) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first)::value;
        // two accumulators a page, the leading products in the one that starts from -m
        float4_t na[TILES][2], ma[TILES][2];
        ask_k(k_half, 0);
#pragma unroll
        for (int at = 0; at < 2 * KK; ++at) {
            if (at + 1 < 2 * KK) ask_k(k_half, at + 1);
            const int pg = at & 1;
#pragma unroll
            for (int b = 0; b < 6; ++b) {
                __builtin_amdgcn_sched_barrier(0);
                const bf16x8_t kv = __builtin_bit_cast(bf16x8_t, op[at][TERMS[b].l]);
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    const bf16x8_t qv = QT == 2 && TERMS[b].r == 2 ? __builtin_bit_cast(bf16x8_t, q2[at >> 1][t])
                                                                   : q[t][at >> 1][TERMS[b].r < QT ? TERMS[b].r : 0];
                    if ((b & 1) == 0) {
                        na[t][pg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv, qv, at < 2 && b == 0 ? neg_m[t] : na[t][pg], 0, 0, 0);
                    } else {
                        const float4_t zero = float4_t{0.f, 0.f, 0.f, 0.f};
                        ma[t][pg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv, qv, at < 2 && b == 1 ? zero : ma[t][pg], 0, 0, 0);
                    }
                }
                const int beat = at * 6 + b;
                if (!FIRST) {
                    constexpr int P_TO = SHARE ? BEATS / 2 : BEATS;
                    const int ps = done_before(beat, 9, 0, P_TO); // at most one step a beat
                    if (done_before(beat + 1, 9, 0, P_TO) > ps) prob_step(ps);
                }
                if (MADE || !FIRST) feed(next, true, beat);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (!FIRST) {
#pragma unroll
                for (int k = 0; k < 3; ++k) p[t][k] = __builtin_bit_cast(bf16x8_t, u4{pw[t][k][0], pw[t][k][1], pw[t][k][2], pw[t][k][3]});
            }
            sa[t] = na[t][0] + ma[t][0];
            sb[t] = na[t][1] + ma[t][1];
        }
    };
    // window 2: accumulation of this group
    auto accumulate = [&](const u4 *v_half, const Item &next) __attribute__((always_inline)) {
        ask_v(v_half, 0);
#pragma unroll
        for (int at = 0; at < NT; ++at) {
            if (at + 1 < NT) ask_v(v_half, at + 1);
#pragma unroll
            for (int b = 0; b < 6; ++b) {
                __builtin_amdgcn_sched_barrier(0);
                const bf16x8_t vv = __builtin_bit_cast(bf16x8_t, op[at][TERMS[b].l]);
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    float4_t &sum = APART && b > 0 ? o_low[t][APART ? at : 0] : o[t][at];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, p[t][TERMS[b].r], sum, 0, 0, 0);
                }
                feed(next, false, at * 6 + b);
                if (MADE && at * 6 + b >= BEATS / 2 && at * 6 + b < BEATS / 2 + 4) top_step(at * 6 + b - BEATS / 2);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // An item is read once its copies have landed, everybody's (a barrier); the copies of the item NBUF - 1 further go out
    // meanwhile, to the buffer that the barrier has freed. With three buffers those of the item between stay in flight.
    constexpr int AHEAD = NBUF == 3 ? CPW : 0;
    // ---- first group's scores
    const Item none{};
    if constexpr (MADE) {
        copies_left<AHEAD>();
    } else {
#pragma unroll
        for (int s = 0; s < SPLIT_STEPS; ++s) split_step(s, false);
        load_k(0, GP);
        if constexpr (!SHARE) load_v(0, 0);
    }
    __syncthreads();
    if constexpr (TOGETHER) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
                for (int k = 0; k < 3; ++k) q[t][kk][k] = __builtin_bit_cast(bf16x8_t, queries[((t * KK + kk) * 3 + k) * 64]);
            }
        }
        if constexpr (!Q_APART) __syncthreads(); // (the next copies go there)
    }
    scores(planes, !MADE ? none : NBUF == 3 ? item_of(0, true, 2) : item_of(1, false, 1), std::true_type{});
    mask(half);
#pragma unroll
    for (int q = 0; q < 4; ++q) top_step(q);
    settle();
    if constexpr (MADE) {
        copies_left<AHEAD>();
    } else {
        __syncthreads();
#pragma unroll
        for (int s = 0; s < SPLIT_STEPS; ++s) split_step(s, false);
        if constexpr (SHARE) load_v(0, 0);
        ask_ids(GP);
    }
    __syncthreads();

    int buf = 1; // MADE: of K of the next group
    auto turned = [&](int b, int n) { return b + n >= NBUF ? b + n - NBUF : b + n; };
    if constexpr (MADE) {
        for (int group = 0; group < n_groups; ++group) {
            const int v_buf = turned(buf, 1);
            scores(planes + buf * ITEM, NBUF == 3 ? item_of(group + 2, false, turned(buf, 2)) : item_of(group, true, v_buf), std::false_type{});
            mask((group + 1) * HALVES + half);
            copies_left<AHEAD>();
            __syncthreads();
            accumulate(planes + v_buf * ITEM, NBUF == 3 ? item_of(group + 1, true, buf) : item_of(group + 2, false, buf));
            settle();
            copies_left<AHEAD>();
            __syncthreads();
            buf = turned(v_buf, 1);
        }
    } else {
        // K of the next group is in LDS, V of this one in registers
        for (int group = 0; group < n_groups; ++group) {
            const int it0 = (group + 1) * GP; // lane 0's entry of ids: the first page of the next group
            mask_v(group * GP);
            if constexpr (!SHARE) load_k(it0, GP);
            scores(planes, none, std::false_type{});
            if constexpr (SHARE) load_k(it0, GP);
            __syncthreads();
            if constexpr (!SHARE) load_v(it0, 0);
            if constexpr (!SHARE) ask_ids(it0 + GP);
            accumulate(v_planes, none);
            if constexpr (SHARE) {
                load_v(it0, 0);
                ask_ids(it0 + GP);
            }
            mask((group + 1) * HALVES + half);
#pragma unroll
            for (int q = 0; q < 4; ++q) top_step(q);
            settle();
            __syncthreads();
        }
    }
    if constexpr (MADE && AHEAD > 0) { // nothing may land in what follows, nor behind the end
        copies_landed();
        if constexpr (HALVES > 1) __syncthreads();
    }

    if constexpr (APART) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int u = 0; u < NT; ++u) o[t][u] += o_low[t][u];
        }
    }

    // ---- the second half's states join the first's through LDS -----------------------------
    if constexpr (HALVES > 1) {
        static_assert(HALVES == 2 && TW * TILES * (NT + 1) * 64 <= NBUF * ITEM, "the second half's states fit the page buffers");
        float4_t *xo = reinterpret_cast<float4_t *>(kv_planes) + (tw * TILES) * (NT + 1) * 64 + lane;
        if (half == 1) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
#pragma unroll
                for (int u = 0; u < NT; ++u) xo[(t * (NT + 1) + u) * 64] = o[t][u];
                xo[(t * (NT + 1) + NT) * 64] = float4_t{thr_i[t] < 0 ? -INFINITY : m_base[t], l_run[t], 0.f, 0.f};
            }
        }
        __syncthreads();
        if (half == 1) return;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float4_t ml = xo[(t * (NT + 1) + NT) * 64];
            const float m0 = thr_i[t] < 0 ? -INFINITY : m_base[t], m1 = ml[0];
            const float mx = fmaxf(m0, m1);
            const float m_safe = mx == -INFINITY ? 0.0f : mx;
            const float w0 = fast_exp2(m0 - m_safe), w1 = fast_exp2(m1 - m_safe);
            l_run[t] = l_run[t] * w0 + ml[1] * w1;
#pragma unroll
            for (int u = 0; u < NT; ++u) o[t][u] = o[t][u] * w0 + xo[(t * (NT + 1) + u) * 64] * w1;
            m_base[t] = m_safe;
            thr_i[t] = mx == -INFINITY ? UNSEEN : SEEN;
        }
    }

    // One slot again, in f32 products, by the whole wavefront. An infinite factor has no three terms (an
    // infinity times its own remainder, or times the second term of the other factor, is NaN), and in V
    // it reaches the slots that do not attend its row as 0 x NaN; so the slots whose sums are not
    // numbers come here, where keys outside the slot's range are left out and an infinity does what it does in
    // f32. What is NaN then stays NaN. Lane (n, j) holds key n's dims 4j .. 4j+3 of every 16, then dim n's keys
    // 4j .. 4j+3. Rare and not fast: a few registers, so that the kernel above keeps its own, and VT tiles of 16
    // dims of V at a time, the scores taken again for each VT.
    const DecodeArgs &args = a;
    const ChunkPages &pages = c;
    const TermPairs &term_pairs = terms;
    auto plain_slot = [&](int slot, float *dst, bool whole, long pidx) {
        // Up to head_dim 128 the arguments come again from the launch's memory: kept in registers for this place
        // they spill around the loop above (this function costs 1500 rows through 4 layers of q32/kv8/hd128,
        // 838 us, 1.2 % so and 0.5 % as it is). At 256, where reading them again makes the compiler spill inside the
        // loop, they are kept (512 rows of q16/kv2/hd256 over 8192 rows: 0.5 %, and 2.7 % with them read again).
        const char *mem = reinterpret_cast<const char *>(&args);
        if constexpr (P <= 128) {
            mem = (const char *)__builtin_amdgcn_kernarg_segment_ptr();
            asm("" : "+s"(mem)); // (not known to be what has been read before)
        }
        const DecodeArgs &a = *reinterpret_cast<const DecodeArgs *>(mem);
        const ChunkPages &c = P <= 128 ? *reinterpret_cast<const ChunkPages *>(mem + sizeof(DecodeArgs)) : pages;
        const TermPairs &tp = P <= 128 ? *reinterpret_cast<const TermPairs *>(mem + sizeof(DecodeArgs) + sizeof(ChunkPages)) : term_pairs;
        static_assert(sizeof(DecodeArgs) % alignof(ChunkPages) == 0 && (sizeof(DecodeArgs) + sizeof(ChunkPages)) % alignof(TermPairs) == 0,
                      "the launch's memory holds the three side by side");
        const Geom &g = a.g;
        auto limit_of = [&](int slot) { return a.q_pos0 + slot_row(a.g, slot); };
        auto ws_of = [&](int slot) { return a.window > 0 ? max(a.window_start, limit_of(slot) + 1 - a.window) : a.window_start; };
        constexpr int VT = NT < 8 ? NT : 8, KT = NT % 4 == 0 ? 4 : NT % 3 == 0 ? 3 : NT;
        static_assert(NT % VT == 0 && NT % KT == 0, "whole steps");
        const float *qrow = a.q + context_row(g, kvh, slot) * g.head_dim;
        const int lo0 = ws_of(slot), hi0 = limit_of(slot);
#pragma unroll 1
        for (int v0 = 0; v0 < NT; v0 += VT) {
            float acc[VT], m = -INFINITY, sum = 0.0f; // sum: of the keys n of every page
#pragma unroll
            for (int u = 0; u < VT; ++u) acc[u] = 0.0f;
#pragma unroll 1
            for (int e = pb0; e < pb1; ++e) {
                const int pos0 = entry_pos<RING>(c, e);
                const int lo = max(lo0, entry_lo<RING>(c, e)), hi = min(hi0, entry_hi<RING>(c, e));
                if (pos0 + 15 < lo || pos0 > hi) continue; // uniform
                const bool own = RING && e >= c.n_old; // a ring's new rows: MADE, in the caller's memory, else in pages of their own
                const uint32_t at = MADE && own ? 0 : entry_tile<RING>(a, c, e, kvh);
                const float4_t *kt = reinterpret_cast<const float4_t *>(!MADE && own ? c.k_new : a.k_pool) + at + lane;
                const float4_t *vt = reinterpret_cast<const float4_t *>(!MADE && own ? c.v_new : a.v_pool) + at + lane + v0 * 64;
                const long kv_dim = (long)g.kv_heads * g.head_dim;
                auto row_at = [&](const float *src, int p) {
                    return src + (long)(min(max(p, tp.new_pos), tp.pos_hi) - tp.new_pos) * kv_dim + (long)kvh * g.head_dim;
                };
                float sc = 0.0f;
#pragma unroll 1
                for (int k0 = 0; k0 < NT; k0 += KT) {
#pragma unroll
                    for (int u = 0; u < KT; ++u) {
                        float4_t x;
                        if (MADE && own) {
                            const float *row = row_at(tp.k_src, pos0 + n);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const int d = (k0 + u) * 16 + j * 4 + i;
                                x[i] = d < g.head_dim ? row[d] : 0.0f;
                            }
                        } else {
                            x = kt[(k0 + u) * 64];
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int d = (k0 + u) * 16 + j * 4 + i;
                            const float y = qrow[min(d, g.head_dim - 1)] * a.qscale;
                            sc += x[i] * (d < g.head_dim ? y : 0.0f); // (K is zero there)
                        }
                    }
                }
                sc = rows_sum(sc);
                sc = pos0 + n >= lo && pos0 + n <= hi ? sc : -INFINITY;
                float top = sc;
#pragma unroll
                for (int x = 1; x < 16; x *= 2) top = fmaxf(top, __shfl_xor(top, x, 64));
                const float m_new = fmaxf(m, top), m_safe = m_new == -INFINITY ? 0.0f : m_new;
                const float alpha = fast_exp2(m - m_safe), pk = fast_exp2(sc - m_safe);
                m = m_new;
                sum = sum * alpha + pk;
#pragma unroll
                for (int u = 0; u < VT; ++u) acc[u] *= alpha;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float pi = __shfl(pk, j * 4 + i, 64);
                    const bool in = pos0 + j * 4 + i >= lo && pos0 + j * 4 + i <= hi;
#pragma unroll
                    for (int u = 0; u < VT; ++u) {
                        const int col = (v0 + u) * 16 + n;
                        const float x = MADE && own ? row_at(tp.v_src, pos0 + j * 4 + i)[min(col, g.head_dim - 1)] : vt[u * 64][i];
                        acc[u] += in ? pi * x : 0.0f;
                    }
                }
                if (__builtin_amdgcn_ballot_w64(sum != sum)) break; // a weight that is NaN: nothing is a number any more
            }
#pragma unroll
            for (int x = 1; x < 16; x *= 2) sum += __shfl_xor(sum, x, 64);
            if (!whole && lane == 0) {
                a.part_m[pidx] = m;
                a.part_l[pidx] = sum;
            }
            // (a NaN sum: the rows that were not looked at any more are NaN too)
            const float scale = whole ? 1.0f / sum : sum != sum ? sum : 1.0f;
#pragma unroll
            for (int u = 0; u < VT; ++u) {
                const float x = rows_sum(acc[u]) * scale;
                const int col = (v0 + u) * 16 + n;
                if (j == 0 && col < g.head_dim) dst[col] = x;
            }
        }
    };

    // ---- every wavefront writes its own slots -------------------------------------------
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const float l = rows_sum(l_run[t]);
        const int slot0 = wg_slot0 + (tw * TILES + t) * 16;
        if (!t_on[t]) continue;
        const bool whole = a.splits_total == 1;
        auto partial_of = [&](int slot) { return ((long)kvh * a.splits_total + a.split_base + split) * n_slots + slot; };
        auto dst_of = [&](int slot) {
            return whole ? a.out + context_row(g, kvh, slot) * g.head_dim
                         : a.part_o + partial_of(slot) * g.head_dim;
        };
        // slots whose sums are not all numbers (columns past head_dim are none of theirs)
        float zero = 0.0f * l;
        if (g.head_dim == P) { // uniform
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                const float4_t z = o[t][u];
                zero = fmaf(z[0], 0.0f, fmaf(z[1], 0.0f, fmaf(z[2], 0.0f, fmaf(z[3], 0.0f, zero))));
            }
        } else {
#pragma unroll
            for (int u = 0; u < NT; ++u) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    zero = fmaf(word_f32(f32_word(o[t][u][i]) & (uint32_t)((u * 16 + j * 4 + i - g.head_dim) >> 31)), 0.0f, zero);
            }
        }
        const uint64_t lanes = __builtin_amdgcn_ballot_w64(!(zero == 0.0f));
        const uint32_t odd = (uint32_t)(lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffffu;
        for (uint32_t left = odd; left; left &= left - 1) {
            const int slot = slot0 + __builtin_ctz(left);
            if (slot < n_slots) plain_slot(slot, dst_of(slot), whole, partial_of(slot));
        }
        const int slot = slot0 + n;
        if (slot >= n_slots || (odd >> n & 1)) continue;
        float *dst = dst_of(slot);
        const float scale = whole ? 1.0f / l : 1.0f;
        if (!whole && j == 0) {
            a.part_m[partial_of(slot)] = thr_i[t] < 0 ? -INFINITY : m_base[t];
            a.part_l[partial_of(slot)] = l;
        }
        const bool vec_ok = (g.head_dim & 3) == 0;
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int col = u * 16 + j * 4;
            const float4_t v = o[t][u] * scale;
            if (vec_ok) {
                if (col < g.head_dim) *reinterpret_cast<float4_t *>(dst + col) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (col + i < g.head_dim) dst[col + i] = v[i];
            }
        }
    }
}

// Query slots of a workgroup; 0 = the kernel does not serve the head_dim.
int f32_prefill_slots(int P, bool halves) { return P > 256 ? 0 : halves && P <= 128 ? 64 : 128; }

size_t f32_terms_bytes(const Geom &g) { return (size_t)g.kv_heads * 2 * 3 * 4 * g.P * sizeof(u4); }

hipError_t launch_f32_terms(const DecodeArgs &a, const ChunkPages &c, const TermPairs &t, hipStream_t s) {
    if (t.held <= 0 || t.entries <= 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)t.held, (unsigned)a.g.kv_heads, (unsigned)(2 * ((4 * a.g.P + 255) / 256)));
    const bool ring = c.ring_pages > 0;
    switch (a.g.P) {
#define SKV_TERMS(P)                                                                              \
    case P:                                                                                       \
        if (ring) hipLaunchKernelGGL((f32_terms_kernel<P, true>), grid, dim3(256), 0, s, a, c, t); \
        else hipLaunchKernelGGL((f32_terms_kernel<P, false>), grid, dim3(256), 0, s, a, c, t);    \
        break
        SKV_TERMS(32);
        SKV_TERMS(64);
        SKV_TERMS(96);
        SKV_TERMS(128);
        SKV_TERMS(256);
#undef SKV_TERMS
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int P, int TILES, int WAVES, int HALVES, bool RING, bool MADE>
static hipError_t launch_f32_prefill_of(const DecodeArgs &a, const ChunkPages &c, const TermPairs &t, dim3 grid, hipStream_t s) {
    constexpr size_t lds = ((size_t)f32_prefill_buffers(P, MADE) * HALVES * 3 * 4 * P + (P > 128 ? WAVES * TILES * (P / 32) * 64 : 0) +
                                   (f32_queries_apart(P, TILES, WAVES, HALVES, MADE) ? f32_query_units(P, TILES, WAVES, HALVES) : 0)) * sizeof(u4);
    static_assert(lds <= 160 * 1024, "a group's K and V (and the queries' third terms) share the LDS of a compute unit");
    static std::atomic<uint64_t> lds_ok{0}; // per instantiation
    {
        hipError_t e = allow_full_lds(reinterpret_cast<const void *>(&f32_prefill_kernel<P, TILES, WAVES, HALVES, RING, MADE>), lds_ok);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((f32_prefill_kernel<P, TILES, WAVES, HALVES, RING, MADE>), grid, dim3(WAVES * 64), lds, s, a, c, t);
    return hipGetLastError();
}
template <int P, int TILES, int WAVES, int HALVES>
static hipError_t launch_f32_prefill_p(const DecodeArgs &a, const ChunkPages &c, const TermPairs *t, dim3 grid, hipStream_t s) {
    if (t) return c.ring_pages > 0 ? launch_f32_prefill_of<P, TILES, WAVES, HALVES, true, true>(a, c, *t, grid, s)
                                   : launch_f32_prefill_of<P, TILES, WAVES, HALVES, false, true>(a, c, *t, grid, s);
    return c.ring_pages > 0 ? launch_f32_prefill_of<P, TILES, WAVES, HALVES, true, false>(a, c, TermPairs{}, grid, s)
                            : launch_f32_prefill_of<P, TILES, WAVES, HALVES, false, false>(a, c, TermPairs{}, grid, s);
}

hipError_t launch_f32_prefill(const DecodeArgs &a, const ChunkPages &c, const TermPairs *t, bool halves, hipStream_t s) {
    const int n_slots = a.n_queries * a.g.gqa;
    const int per_wg = f32_prefill_slots(a.g.P, halves);
    if (per_wg == 0) return hipErrorInvalidValue;
    halves = per_wg == 64;
    dim3 grid((unsigned)a.splits, (unsigned)a.g.kv_heads, (unsigned)((n_slots + per_wg - 1) / per_wg));
    switch (a.g.P) {
    case 32: return halves ? launch_f32_prefill_p<32, 1, 8, 2>(a, c, t, grid, s) : launch_f32_prefill_p<32, 1, 8, 1>(a, c, t, grid, s);
    case 64: return halves ? launch_f32_prefill_p<64, 1, 8, 2>(a, c, t, grid, s) : launch_f32_prefill_p<64, 1, 8, 1>(a, c, t, grid, s);
    case 96: return halves ? launch_f32_prefill_p<96, 1, 8, 2>(a, c, t, grid, s) : launch_f32_prefill_p<96, 1, 8, 1>(a, c, t, grid, s);
    case 128: return halves ? launch_f32_prefill_p<128, 1, 8, 2>(a, c, t, grid, s) : launch_f32_prefill_p<128, 1, 8, 1>(a, c, t, grid, s);
    case 256: return launch_f32_prefill_p<256, 1, 8, 1>(a, c, t, grid, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace skv

// gfx950 kernels of the KV hot path, part 3: chunked prefill over the paged cache, the one
// matrix-core-bound kernel of the path.
#include <type_traits>

#include "append_tile.h"
#include "chunk_pages.h"
#include "lds_copy.h"

namespace skv {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) short short4_t;
typedef __attribute__((ext_vector_type(4))) float float4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u4;

namespace {

// two values rounded to bf16 (nearest even), the first in the low half: one instruction
__device__ __forceinline__ uint32_t bf16_pair(float x, float y) {
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, b2));
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

} // namespace

// ------------------------------------------------------------------------------------
// Many query rows over the cache (cached_attention_prefill_rows,
// src/decoder/attention_ops.rs:976-1017, as one launch): query slot (i, g) = new row i,
// head g of the kv head's group, attends positions up to q_pos0 + i through the layer's window.
//
// One workgroup = WAVES wavefronts of TILES tiles of 16 query slots of one kv head, and a range
// of the pages any of them attends (split). The workgroup walks its pages once, in pairs: all
// threads copy the pages' K and V tiles (already in matrix-operand order) from memory to LDS,
// double buffered, and every wavefront multiplies them with its own query tiles, which it holds
// in registers as bf16 hi + lo halves (pre-scaled by log2(e)/sqrt(head_dim)). Per pair:
//   window 1: S^T(p+1) = K . Q^T of the NEXT pair (16x16x32 products over the head dims) with the
//             exponentials and the hi + lo split of this pair's probabilities between the products;
//   window 2: O^T += V^T . P^T(p), 16x16x32 products over the pair's 32 keys, with the next operands' halves put side by
//             side and the search for the largest of the next pair's scores between the products.
// A product occupies the matrix pipe for 16 cycles and its wavefront for 4; the vector work of
// the softmax therefore costs nothing where it is issued between products that do not depend on
// it, and a pair's softmax never depends on the next pair's scores. (With the softmax between the
// two products of the same pair, the two wavefronts of a SIMD, which a barrier keeps in step,
// were in their vector phases at the same time: four pairs at head_dim 128 took 4.4 us by
// time stamps where they take 3.4 now, of which the products are 1.75.)
//
// The softmax runs in base 2 against a base m per slot that is not the running maximum but up to 4
// above it: the score accumulators start at -m, so the products deliver s - m and the exponential
// needs no subtraction, and only a score above m makes the wavefront move the bases (to 4 above that
// score) and rescale its sums. Probabilities are at most one, so that sums of large values are no larger
// than against the maximum, and are split relatively, so nothing is lost; partials carry (o, base, l) and any
// base serves the merge. (A step of 2 moves the bases more often, 1.5 % of a prompt; one of 8 is no faster, and
// accumulators that start further from zero are less exact: 2 % more error against 64 bits.)
// With HALVES = 2 (or 4) the wavefronts are two halves (four quarters) that hold the same slots and take
// the page pairs in turn; the others' (o, m, l) join the first's through LDS at the end. Otherwise there is
// no merge inside the workgroup; with several splits the partials go to merge_rows_kernel.
// The copies go straight from memory to LDS. 512 rows as one call (append, attention, merge), in us
// on one MI355X, against the kernel that ran scores, softmax and accumulation of a pair one after
// the other and copied through registers: q32/kv8/hd128 over 0, 1536, 4700, 16384 rows 34.5 -> 21.7,
// 57.2 -> 41.1, 106 -> 86.5, 256 -> 225; q16/kv2/hd256 40.0 -> 24.3, 55.7 -> 50.5, 97.9 -> 89.0, 247 -> 225 (where
// the matrix pipes alone need 130).
// A wavefront issues an instruction in four to five cycles, so every one beside the products counts: with a tile per
// wavefront to copy and the moves that put operands together and the search for the maximum between products, chunks of 512
// rows on layers that are in no cache went, in us, for q32/kv8/hd128 over 4700, 16384 from 88.0 to 80.5, 224 to 213; for
// q16/kv8/hd256 on a ring of 1024 rows from 47.2 to 44.1. (Second terms of the probabilities as dot products of the pair of
// first terms with -1 and 0, an instruction less each, took longer: 1024 rows of q24/kv8/hd128 over 4000 139.4 against 132.2. Three
// wavefronts per SIMD, twelve in thirds at 154 registers, were no faster than two; two tiles per wavefront at head_dim 256, four
// wavefronts at 400 registers, 11 to 40 % slower.)
// ------------------------------------------------------------------------------------

// LDS order of a step, SP pairs: [SP][K tile of page A | K tile of page B], then V the same way, tiles
// as they are in memory.
//
// Keys that no query slot of the workgroup attends (rows at or past the cache's length after a
// rollback, ring rows not valid, rows before every slot's window, the stand-in page past the
// end of a split) get zero probability, but 0 x NaN is NaN: in steps that touch the edges of the
// attended range their V values are cleared in LDS, behind a barrier of its own, so the bits of
// such a row never reach a context (the reference never reads those rows,
// src/decode_resident/kernels.rs:11-88).
// 16-byte units of LDS: two buffers of a step's pages, [K of SP pairs | V of SP pairs] each. The parts of a workgroup, which hold the same
// query tiles, make their operands together (QUERIES units, behind the first group's K in the second buffer).
template <int P, int TILES, int SP, int WAVES, int HALVES>
struct TileLds {
    static constexpr int KK = P / 32, TILE = KK * 64, GP = 2 * HALVES;
    static constexpr int BUF = 2 * SP * GP * TILE;
    static constexpr bool TOGETHER = HALVES > 1 && KK > 1;
    static constexpr int QUERIES_AT = BUF + GP * TILE, QUERIES = TOGETHER ? WAVES / HALVES * TILES * KK * 2 * 64 : 0;
    static constexpr int UNITS = 2 * BUF > QUERIES_AT + QUERIES ? 2 * BUF : QUERIES_AT + QUERIES;
};

template <int P, int TILES, int SP, int WAVES, int HALVES, bool RING>
__global__ __launch_bounds__(WAVES * 64) void prefill_tile_kernel(DecodeArgs a, ChunkPages c) {
    constexpr int THREADS = WAVES * 64;
    constexpr int KK = P / 32;
    constexpr int NT = P / 16;
    // Vector work is held in its place between the products; a wavefront alone on its SIMD (head_dim above 256), and one with
    // few products to a pair (up to 96), does better where the compiler places it (256 rows of q8/kv2/hd512 over 4096: 61.0 us
    // against 66.0; 1024 of q8/kv2/hd64 over 8000: 53.0 against 55.7; heads of 65 to 96 dims 1 to 3 %)
    constexpr bool PINNED = KK >= 4 && P <= 256;
    constexpr int TILE_U4 = KK * 64;                           // 16-byte units of one K (or V) tile
    constexpr int GP = 2 * HALVES;                             // pages of a group: a pair for each half
    static_assert(TILE_U4 % 64 == 0, "a wavefront copies whole KiB of one page");
    extern __shared__ __attribute__((aligned(16))) u4 kv_lds[]; // [2 buffers][K of SP pairs | V of SP pairs]
    constexpr int HALF_U4 = SP * GP * TILE_U4;
    constexpr int BUF_U4 = 2 * HALF_U4;

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
    constexpr int TW = WAVES / HALVES;                         // wavefronts of a half, TILES slot tiles each
    const int half = HALVES > 1 ? wave / TW : 0;
    const int tw = HALVES > 1 ? wave % TW : wave;
    const int wg_slot0 = blockIdx.z * (TW * TILES * 16);
    const int wg_slot1 = min(n_slots, wg_slot0 + TW * TILES * 16) - 1; // last slot of the workgroup

    // query slot -> position of its row (the last it attends), first position it attends
    auto limit_of = [&](int slot) { return a.q_pos0 + slot_row(a.g, slot); };
    auto ws_of = [&](int slot) { return a.window > 0 ? max(a.window_start, limit_of(slot) + 1 - a.window) : a.window_start; };

    // entries of the page list any slot of the workgroup can see, divided among the splits
    const int wg_ws_lo = ws_of(wg_slot0);
    const int wg_lim_hi = limit_of(wg_slot1);
    auto entry_of = [&](int pos) {
        if (!RING) return pos >> 4;
        return pos < c.new_pos0 ? max((pos - c.first_pos) >> 4, 0) : c.n_old + ((pos - c.new_first) >> 4);
    };
    const int e_lo = entry_of(wg_ws_lo);
    const int e_hi = entry_of(wg_lim_hi) + 1;
    const unsigned span = (unsigned)(e_hi - e_lo);
    const int pb0 = e_lo + (int)(((unsigned)split * span) / (unsigned)a.splits);
    const int pb1 = e_lo + (int)(((unsigned)(split + 1) * span) / (unsigned)a.splits);
    const int n_it = pb1 - pb0;
    const int n_groups = (n_it + GP - 1) / GP;

    // ---- page copies, memory -> LDS. K runs one group ahead of V: step s brings K of the groups
    // SP*s + 1 .. and V of the groups SP*s ..
    auto entry = [&](int it) { return min(pb0 + it, e_hi - 1); }; // past the end: a page again, unused
    // Places of the next copy's tiles, one per lane, asked for a step ahead and read with
    // v_readlane: a scalar read of the table in front of the loads would make the wavefront wait
    // for it and, the two being counted together, for every LDS read in flight (512 rows of
    // q16/kv2/hd256 over 16384 rows: 285 us against 265).
    uint32_t ids;
    auto ask_ids = [&](int it) __attribute__((always_inline)) { ids = entry_tile<RING>(a, c, entry(it + lane), kvh); };
    // tile of page it0 + d, it0 being the page that lane 0's entry belongs to
    auto tile_of = [&](int it0, int d, bool v) __attribute__((always_inline)) {
        const uint16_t *pool = v ? a.v_pool : a.k_pool;
        if (RING && entry(it0 + d) >= c.n_old) pool = v ? c.v_new : c.k_new;
        return reinterpret_cast<const u4 *>(pool) + (uint32_t)__builtin_amdgcn_readlane(ids, d);
    };
    ask_ids(0);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)kv_lds;
    const uint32_t lane_at = (uint32_t)lane * 16;
    // A wavefront copies whole tiles, TPW of a step's K and then V tiles, a KiB an instruction: one place in the page
    // list and one address for four instructions (with the KiBs of a step dealt out to the wavefronts in turn, each had
    // a place, an address and an LDS address of its own: nine instructions a copy, seventy of a step's four hundred).
    constexpr int TPW = 2 * SP * GP / WAVES, CPT = TILE_U4 / 64;
    static_assert(2 * SP * GP % WAVES == 0, "a wavefront copies whole tiles");
    const u4 *from[TPW];
    auto find_tiles = [&](int it0) __attribute__((always_inline)) { // it0: see tile_of; the step's first V page
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            const int ti = wave * TPW + i;
            const bool v = ti >= SP * GP;
            from[i] = tile_of(it0, v ? ti - SP * GP : ti + GP, v);
        }
    };
    // KiB i of the wavefront's copies, to the buffer half at unit `dst` of LDS
    auto copy_kib = [&](int i, int dst) __attribute__((always_inline)) {
        const int quad = i % CPT / 4 * 256;
        copy_to_lds(from[i / CPT] + quad, lane_at, lds0 + (uint32_t)(dst + (wave * TPW + i / CPT) * TILE_U4 + quad) * 16, i % CPT % 4);
    };
    // The copies of a step are spread over the K-steps of the first half of its products (512 rows of
    // q16/kv2/hd256 over 16384 rows: 243 us against 265 with all of them in front of one window; 223
    // with copies straight to LDS instead of through registers, which took stores besides).
    constexpr int COPY_SPAN = KK * SP;
    auto copy_slot = [&](int slot, int step) __attribute__((always_inline)) {
        if (slot == 0) {
            find_tiles((step + 1) * SP * GP); // first page of the V copy, a group before the K copy's
            ask_ids((step + 2) * SP * GP);
        }
#pragma unroll
        for (int i = 0; i < TPW * CPT; ++i)
            if (i * COPY_SPAN / (TPW * CPT) == slot) copy_kib(i, ((step + 1) & 1) * BUF_U4);
    };
    // V rows of the pages from first_page on that nobody attends, cleared in the buffer half at `v`
    const Inner wg_in = inner_entries<RING>(c, pb0, pb1, wg_ws_lo, wg_lim_hi);
    auto clear_v = [&](int first_page, u4 *v) __attribute__((always_inline)) {
        const int e0 = pb0 + first_page, e1 = e0 + SP * GP;
        if ((e0 >= wg_in.o0 && e1 <= wg_in.o1) || (RING && e0 >= wg_in.n0 && e1 <= wg_in.n1)) return; // uniform
        for (int i = tid; i < SP * GP * TILE_U4; i += THREADS) {
            const int it = first_page + i / TILE_U4;
            const int e = entry(it);
            const int pos0 = entry_pos<RING>(c, e) + ((i >> 4) & 3) * 4; // unit: keys 4rq .. 4rq+3 of two dims
            const int lo = max(wg_ws_lo, entry_lo<RING>(c, e)), hi = min(wg_lim_hi, entry_hi<RING>(c, e));
            uint32_t keep[2] = {0u, 0u};
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (it < n_it && pos0 + r >= lo && pos0 + r <= hi) keep[r >> 1] |= 0xffffu << ((r & 1) * 16);
            v[i] &= u4{keep[0], keep[1], keep[0], keep[1]};
        }
        __syncthreads();
    };

    // ---- this wavefront's query tiles ------------------------------------------------
    int my_limit[TILES], my_ws[TILES];
    int t_ws_hi[TILES], t_lim_lo[TILES]; // per tile extremes
    bool t_on[TILES];
    bf16x8_t qh[TILES][KK], ql[TILES][KK];
    // The parts load a share of their tiles' K-steps each and find the others' in LDS behind the first barrier. (A load whose lanes all
    // hit lines of their own takes 64 cycles; with all of them loaded by every wavefront, 128 such loads a compute unit at
    // head_dim 256, chunks of 512 rows took, in us: q16/kv8/hd256 on a ring 44.5 against 42.0, q32/kv8/hd128 over 0, 1024, 4700
    // 18.3/17.2, 34.5/33.3, 80.7/78.4.)
    using Lds = TileLds<P, TILES, SP, WAVES, HALVES>;
    constexpr int QK = Lds::TOGETHER ? (KK + HALVES - 1) / HALVES : KK; // K-steps of a tile that this wavefront loads
    auto share = [&](int i) { return Lds::TOGETHER ? min(half * QK + i, KK - 1) : i; }; // (the last part may make one again)
    float qv[TILES][QK][8];
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
        // eight consecutive dims of the slot's row per k-step: all loads first (two 16-byte
        // loads per step when the row allows), unconditional from clamped addresses, so that
        // they are one round trip; dims past head_dim are zeroed afterwards
        if (a.q_vec) {
#pragma unroll
            for (int kk = 0; kk < QK; ++kk) {
                const int d0 = share(kk) * 32 + j * 8;
                const float4_t *qp = reinterpret_cast<const float4_t *>(qrow + min(d0, g.head_dim - 8));
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
    u4 *const queries = kv_lds + Lds::QUERIES_AT + tw * TILES * KK * 2 * 64 + lane; // of this wavefront's tiles
    // the first group's K, into the second buffer
#pragma unroll
    for (int u = 0; u < (GP * TILE_U4 + THREADS - 1) / THREADS; ++u) {
        const int i0 = wave * 64 + u * THREADS;
        if (GP * TILE_U4 % THREADS == 0 || i0 < GP * TILE_U4)
            copy_to_lds(tile_of(0, i0 / TILE_U4, false) + i0 % TILE_U4, lane_at, lds0 + (uint32_t)(BUF_U4 + i0) * 16);
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int kk = 0; kk < QK; ++kk) {
            const int d0 = share(kk) * 32 + j * 8;
            uint32_t hi[4], lo[4];
            // (with 16-byte loads head_dim is a multiple of 8: the lane's eight dims are all inside or all padding)
            const float scale = !a.q_vec || d0 < g.head_dim ? a.qscale : 0.0f;
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) {
                float x0 = qv[t][kk][e2 * 2] * scale, x1 = qv[t][kk][e2 * 2 + 1] * scale;
                if (!a.q_vec) {
                    x0 = d0 + e2 * 2 < g.head_dim ? x0 : 0.0f;
                    x1 = d0 + e2 * 2 + 1 < g.head_dim ? x1 : 0.0f;
                }
                hi[e2] = bf16_pair(x0, x1);
                lo[e2] = bf16_pair(x0 - __uint_as_float(hi[e2] << 16), x1 - __uint_as_float(hi[e2] & 0xffff0000u));
            }
            if constexpr (Lds::TOGETHER) {
                u4 *at = queries + (t * KK + share(kk)) * 2 * 64;
                at[0] = u4{hi[0], hi[1], hi[2], hi[3]};
                at[64] = u4{lo[0], lo[1], lo[2], lo[3]};
            } else {
                qh[t][kk] = __builtin_bit_cast(bf16x8_t, u4{hi[0], hi[1], hi[2], hi[3]});
                ql[t][kk] = __builtin_bit_cast(bf16x8_t, u4{lo[0], lo[1], lo[2], lo[3]});
            }
        }
    }
    // The first scores wait for the queries and that K alone; the first step's pages are on their way meanwhile. (The compiler
    // waits for the queries as if there were no copies behind them: with all copies in front of the queries, that wait
    // was for the last page. First scores done, in us after a launch's start: q32/kv8/hd128 over 1024 5.4 -> 5.0,
    // q16/kv8/hd256 on a ring 9.6 -> 8.3; whole chunks of 512 rows 39.7 -> 38.8 over 1536 and 44.3 -> 43.9.)
    copies_landed();
    find_tiles(0);
#pragma unroll
    for (int i = 0; i < TPW * CPT; ++i) copy_kib(i, 0);
    ask_ids(SP * GP);

    float4_t o[TILES][NT];
    float4_t neg_m[TILES];             // -m in all four: what the score accumulators start from
    // base of the slot; a score whose bits reach thr_i moves it: SEEN (any above the base), or, for a slot without a key
    // so far, UNSEEN (whatever it is)
    constexpr int UNSEEN = INT32_MIN, SEEN = 1;
    float m_base[TILES];
    int thr_i[TILES];
    float l_run[TILES];                // this lane's share of the slot's sum
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
        for (int u = 0; u < NT; ++u) o[t][u] = float4_t{0.f, 0.f, 0.f, 0.f};
        m_base[t] = 0.0f;
        neg_m[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        thr_i[t] = UNSEEN;
        l_run[t] = 0.0f;
    }

    // S^T - m of a pair, eight scores a lane and tile: keys 4j .. 4j+3 of page A, then of page B
    float4_t sa[TILES], sb[TILES];
    // probabilities of the pair being accumulated, as two bf16 terms
    bf16x8_t ph[TILES], pl[TILES];
    // K-steps an operand is asked for ahead of its products (of V's a step more, which the moves take)
    constexpr int DEPTH = KK < 2 || TILES > 1 ? 1 : 2;
    constexpr int DEPTH_V = KK < 4 || P > 256 ? DEPTH : DEPTH + 1;

    // the half's pairs are the page pairs HALVES * group + half.
    // pairs whose keys every slot of the wavefront attends: [in0, in1) and, of new pages, [in2, in3)
    int in0, in1, in2, in3;
    {
        int lo = t_ws_hi[0], hi = t_lim_lo[0];
#pragma unroll
        for (int t = 1; t < TILES; ++t) {
            lo = max(lo, t_ws_hi[t]);
            hi = min(hi, t_lim_lo[t]);
        }
        const Inner r = inner_entries<RING>(c, pb0, pb1, lo, hi);
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
    // Whether a score is above its slot's base is whether the largest of the scores' bits, as integers, is positive (a
    // positive float is a positive integer, and every other one is zero or negative): v_max3_i32, where maxima of
    // floats cost an instruction more per operand, to quiet what is no number.
    int mi[TILES];
    auto top_step = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float4_t &x = q < 2 ? sa[t] : sb[t];
            const int m = max(__float_as_int(x[q & 1 ? 2 : 0]), __float_as_int(x[q & 1 ? 3 : 1]));
            mi[t] = q == 0 ? m : max(m, mi[t]);
        }
    };
    // where a score passes the base, the wavefront's bases move
    auto settle = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (__builtin_amdgcn_ballot_w64(mi[t] >= thr_i[t])) {
                const float mx = fmaxf(fmaxf(fmaxf(sa[t][0], sa[t][1]), fmaxf(sa[t][2], sa[t][3])),
                                       fmaxf(fmaxf(sb[t][0], sb[t][1]), fmaxf(sb[t][2], sb[t][3])));
                const float top = rows_max(mx); // of the slot, relative to its base
                const bool unseen = thr_i[t] < 0;
                const float d = top > (unseen ? -INFINITY : 0.0f) ? top + 4.0f : 0.0f;
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
                }
            }
        }
    };

    // probabilities of the settled scores, in nine small steps per tile so that they can stand
    // between products: step q takes the exponential of score q and splits that of score q - 1
    float pr_[TILES];                  // exponential of the last step
    float pr2[TILES][2];
    uint32_t hi4[TILES][4], lo4[TILES][4];
    auto prob_step = [&](int q) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const float prev = pr_[t];
            if (q < 8) pr_[t] = fast_exp2(q < 4 ? sa[t][q & 3] : sb[t][q & 3]);
            if (q > 0) {
                const int e = q - 1;
                l_run[t] += prev;
                pr2[t][e & 1] = prev;
                // p = hi + lo, both rounded to nearest: 2^-18 relative, of either sign (512 rows of q8/kv2/hd64 over 2500: errors of 3.4e-6
                // against 64 bits; with hi the upper 16 bits of p, cut off, as fast, 5.3e-6; both cut off, always too small, 9.9e-6)
                if (e & 1) {
                    const uint32_t hi = bf16_pair(pr2[t][0], prev);
                    hi4[t][e >> 1] = hi;
                    lo4[t][e >> 1] = bf16_pair(pr2[t][0] - __uint_as_float(hi << 16), prev - __uint_as_float(hi & 0xffff0000u));
                    if (PINNED) asm volatile("" : "+v"(hi4[t][e >> 1]), "+v"(lo4[t][e >> 1])); // (here, between the products, not behind them)
                }
            }
        }
    };
    auto probs_done = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            ph[t] = __builtin_bit_cast(bf16x8_t, u4{hi4[t][0], hi4[t][1], hi4[t][2], hi4[t][3]});
            pl[t] = __builtin_bit_cast(bf16x8_t, u4{lo4[t][0], lo4[t][1], lo4[t][2], lo4[t][3]});
        }
    };
    u4 ra[KK], rb[KK];
    auto ask_k = [&](const u4 *kt, int kk) __attribute__((always_inline)) {
        ra[kk] = kt[kk * 64 + lane];
        rb[kk] = kt[TILE_U4 + kk * 64 + lane];
    };
    u4 rva[KK], rvb[KK];
    auto ask_v = [&](const u4 *vt, int kk) __attribute__((always_inline)) {
        rva[kk] = vt[kk * 64 + lane];
        rvb[kk] = vt[TILE_U4 + kk * 64 + lane];
    };
    // window 1: scores of the pair whose K tiles lie at kt (its first operands asked for already),
    // between them the probabilities of the settled pair; the first V operands of `vt` at the end
    auto scores = [&](const u4 *kt, const u4 *vt, auto with_probs, auto copies) __attribute__((always_inline)) {
        constexpr bool PROBS = decltype(with_probs)::value;
        constexpr int BEATS = 2 * KK; // (k-step, hi or lo half)
        // The SIMD's other wavefront may be in its second window, which is products almost alone and so gets on with the cycles that
        // are left (1024 rows of q24/kv8/hd128 over 4000 132.2 -> 128.9 us, of q8/kv2/hd64 over 8000 51.7 -> 50.0; 512 of
        // q32/kv8/hd128 over 16384 212 -> 208; raised in the second window instead: half of that)
        __builtin_amdgcn_s_setprio(1);
        float4_t na[TILES], nb[TILES];
        int q = 0;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            if (kk + DEPTH < KK) ask_k(kt, kk + DEPTH);
            copies(kk);
            if (PROBS && kk + DEPTH_V >= KK) ask_v(vt, kk + DEPTH_V - KK);
            const bf16x8_t ka = __builtin_bit_cast(bf16x8_t, ra[kk]);
            const bf16x8_t kb = __builtin_bit_cast(bf16x8_t, rb[kk]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    const bf16x8_t qv = h ? ql[t][kk] : qh[t][kk];
                    na[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka, qv, kk + h == 0 ? neg_m[t] : na[t], 0, 0, 0);
                    nb[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb, qv, kk + h == 0 ? neg_m[t] : nb[t], 0, 0, 0);
                }
                if (PROBS) {
                    // steps done by the end of this beat
                    const int until = ((kk * 2 + h + 1) * 9) / BEATS;
#pragma unroll
                    for (int k = 0; k < 9; ++k)
                        if (k >= q && k < until) prob_step(k);
                    q = until;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
        if (PROBS) probs_done();
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (PROBS && PINNED) asm volatile("" : "+v"(l_run[t])); // (the sum's additions stay between the products)
            sa[t] = na[t];
            sb[t] = nb[t];
        }
    };
    // A lane's unit holds four keys of dims n and n + 16: both pages' halves side by side are the 32-key operands of
    // the two dim tiles.
    auto v_first = [&](int kk, bf16x8_t &v) __attribute__((always_inline)) {
        u4 x = {rva[kk].x, rva[kk].y, rvb[kk].x, rvb[kk].y};
        if (PINNED) asm volatile("" : "+v"(x)); // (put together here, not in front of the product that takes it)
        v = __builtin_bit_cast(bf16x8_t, x);
    };
    auto v_second = [&](int kk, bf16x8_t &v) __attribute__((always_inline)) {
        u4 x = {rva[kk].z, rva[kk].w, rvb[kk].z, rvb[kk].w};
        if (PINNED) asm volatile("" : "+v"(x));
        v = __builtin_bit_cast(bf16x8_t, x);
    };
    // window 2: O^T += V^T . P^T over the 32 keys of the pair; between the products the next operands are put
    // together and the largest of the settled pair's scores is found
    auto accumulate = [&](const u4 *vt, auto copies) __attribute__((always_inline)) {
        auto fence = [&]() __attribute__((always_inline)) {
            if (PINNED) __builtin_amdgcn_sched_barrier(0);
        };
        bf16x8_t v0, v1, w0, w1;
        v_first(0, v0);
        v_second(0, v1);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            if (kk + DEPTH_V < KK) ask_v(vt, kk + DEPTH_V);
            copies(kk);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    const bf16x8_t pt = h ? pl[t] : ph[t];
                    fence();
                    o[t][2 * kk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v0, pt, o[t][2 * kk], 0, 0, 0);
                    fence();
                    if (h == 0 && t == 0 && kk + 1 < KK) v_first(kk + 1, w0);
                    if (h == 1 && t == 0) {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (PINNED && q * KK / 4 == kk) top_step(q);
                    }
                    fence();
                    o[t][2 * kk + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v1, pt, o[t][2 * kk + 1], 0, 0, 0);
                    fence();
                    if (h == 0 && t == 0 && kk + 1 < KK) v_second(kk + 1, w1);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            v0 = w0;
            v1 = w1;
        }
    };

    // ---- first pair's scores
    const int n_steps = (n_groups + SP - 1) / SP;
    __syncthreads();
    if constexpr (Lds::TOGETHER) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                qh[t][kk] = __builtin_bit_cast(bf16x8_t, queries[(t * KK + kk) * 2 * 64]);
                ql[t][kk] = __builtin_bit_cast(bf16x8_t, queries[(t * KK + kk) * 2 * 64 + 64]);
            }
        }
    }
#pragma unroll
    for (int kk = 0; kk < DEPTH; ++kk) ask_k(kv_lds + BUF_U4 + half * 2 * TILE_U4, kk);
    scores(kv_lds + BUF_U4 + half * 2 * TILE_U4, nullptr, std::false_type{}, [](int) {});
    mask(half);
#pragma unroll
    for (int q = 0; q < 4; ++q) top_step(q);
    settle();
    copies_landed();
    __syncthreads(); // the second buffer is free, the first one full
    clear_v(0, kv_lds + HALF_U4);

    for (int step = 0; step < n_steps; ++step) {
        const u4 *buf = kv_lds + (step & 1) * BUF_U4;
#pragma unroll
        for (int pp = 0; pp < SP; ++pp) {
            const int group = step * SP + pp;
            if (group >= n_groups) continue; // uniform
            const u4 *kt = buf + (pp * HALVES + half) * 2 * TILE_U4;
            const u4 *vt = kt + HALF_U4;
#pragma unroll
            for (int kk = 0; kk < DEPTH; ++kk) ask_k(kt, kk);
            // (after the last step the copies re-read its pages into the idle buffer)
            scores(kt, vt, std::true_type{}, [&](int kk) __attribute__((always_inline)) { copy_slot(2 * KK * pp + kk, step); });
            if (PINNED) mask((group + 1) * HALVES + half);
            accumulate(vt, [&](int kk) __attribute__((always_inline)) { copy_slot(2 * KK * pp + KK + kk, step); });
            if (!PINNED) {
                mask((group + 1) * HALVES + half);
#pragma unroll
                for (int q = 0; q < 4; ++q) top_step(q);
            }
            settle();
        }
        copies_landed();
        __syncthreads();
        if (step + 1 < n_steps) clear_v((step + 1) * SP * GP, kv_lds + ((step + 1) & 1) * BUF_U4 + HALF_U4);
    }

    // ---- the parts join their states through LDS, each the columns that it then stores: part p the tiles u of 16 dims with
    // owner(u) == p. (Quarters with all states joined and stored by the first part's wavefronts:
    // 512 rows of q32/kv8/hd128 over 4700 75.9 us against 75.2. Of halves the first one's do it all: divided, with more of LDS read and written
    // at once, 16 x 256 on a ring takes 38.3 against 38.0.)
    const auto owner = [](int u) { return HALVES == 2 ? 0 : u * HALVES / NT; };
    if constexpr (HALVES > 1) {
        constexpr int SETS = NT * (HALVES - 1) + HALVES; // of a tile: every u from the parts that do not own it; (m, l) of all
        static_assert(TW * TILES * SETS * 64 <= 2 * BUF_U4, "the states fit the page buffers");
        float4_t *xo = reinterpret_cast<float4_t *>(kv_lds) + (tw * TILES) * SETS * 64 + lane; // (the loop ends in a barrier)
        const auto at = [&](int t, int u, int part) { return (t * SETS + u * (HALVES - 1) + (part < owner(u) ? part : part - 1)) * 64; };
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int u = 0; u < NT; ++u)
                if (owner(u) != half) xo[at(t, u, half)] = o[t][u];
            xo[(t * SETS + NT * (HALVES - 1) + half) * 64] = float4_t{thr_i[t] < 0 ? -INFINITY : m_base[t], l_run[t], 0.f, 0.f};
        }
        __syncthreads();
        if (HALVES == 2 && half > 0) return;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            float w[HALVES], l[HALVES], mx = -INFINITY;
#pragma unroll
            for (int h = 0; h < HALVES; ++h) {
                const float4_t ml = xo[(t * SETS + NT * (HALVES - 1) + h) * 64];
                w[h] = ml[0];
                l[h] = ml[1];
                mx = fmaxf(mx, w[h]);
            }
            const float m_safe = mx == -INFINITY ? 0.0f : mx;
            l_run[t] = 0.0f;
#pragma unroll
            for (int h = 0; h < HALVES; ++h) {
                w[h] = fast_exp2(w[h] - m_safe);
                l_run[t] += l[h] * w[h];
            }
            m_base[t] = m_safe;
            thr_i[t] = mx == -INFINITY ? UNSEEN : SEEN;
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                if (owner(u) != half) continue; // uniform
                float4_t sum = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int h = 0; h < HALVES; ++h) sum += (h == owner(u) ? o[t][u] : xo[at(t, u, h)]) * w[h];
                o[t][u] = sum;
            }
        }
    }

    // ---- every wavefront writes its own slots -------------------------------------------
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const float l = rows_sum(l_run[t]);
        const int slot = wg_slot0 + (tw * TILES + t) * 16 + n;
        if (!t_on[t] || slot >= n_slots) continue;
        float *dst;
        float scale = 1.0f;
        if (a.splits_total == 1) {
            scale = 1.0f / l;
            dst = a.out + context_row(g, kvh, slot) * g.head_dim;
        } else {
            const long pidx = ((long)kvh * a.splits_total + a.split_base + split) * n_slots + slot;
            dst = a.part_o + pidx * g.head_dim;
            if (j == 0 && half == 0) {
                a.part_m[pidx] = thr_i[t] < 0 ? -INFINITY : m_base[t];
                a.part_l[pidx] = l;
            }
        }
        const bool vec_ok = (g.head_dim & 3) == 0;
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            if (owner(u) != half) continue; // uniform
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

// Merge of the split partials of many query slots: one thread per (kv head, slot, four
// columns) walks the few splits. (The decode merge spends a workgroup per 16 columns of a
// head, which is right for a handful of heads and many splits, not for thousands of slots.)
// (32-bit indexes inside a kv head, whose slots times columns stay far below 2^31: three 64-bit divisions a
// thread were a quarter of the launch.)
// SPLITS: how many there are, up to four (0: any number): one trip to memory, and nothing is asked for twice. With four loads of
// each kind whatever the number, and the context stored 4 bytes at a time: two splits of 512 rows of q16/kv8/hd256, with the ring append in the
// same launch, 10.6 -> 7.7 us (4.9 TB/s of 38 MB), four of q16/kv2/hd256 9.0 -> 8.2 (5.1 of 42).
template <int SPLITS>
__device__ __forceinline__ void merge_rows_of(const DecodeArgs &a, const int kvh, const int slot, const int c4) {
    const Geom g = a.g;
    const int n_slots = a.n_queries * g.gqa;
    const long base = ((long)kvh * a.splits_total) * n_slots + slot;
    // More than four splits take a pass over m first.
    float mx = -INFINITY;
    if constexpr (SPLITS == 0)
        for (int sp = 0; sp < a.splits_total; ++sp) mx = fmaxf(mx, a.part_m[base + (long)sp * n_slots]);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    float lsum = 0.0f;
    const bool vec_ok = (g.head_dim & 3) == 0;
    // four splits per round: their loads are all issued before the first is consumed (the
    // partials are read once: non-temporal)
    constexpr int N = SPLITS ? SPLITS : 4;
    for (int sp0 = 0; sp0 < (SPLITS ? 1 : a.splits_total); sp0 += N) {
        float w[N], lp[N];
        float4_t v[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int sp = SPLITS ? u : min(sp0 + u, a.splits_total - 1); // a repeat of the last one is left out below
            const long pidx = base + (long)sp * n_slots;
            w[u] = a.part_m[pidx];
            lp[u] = a.part_l[pidx];
            const float *po = a.part_o + pidx * g.head_dim + c4;
            if (vec_ok) {
                v[u] = __builtin_nontemporal_load(reinterpret_cast<const float4_t *>(po));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[u][i] = c4 + i < g.head_dim ? po[i] : 0.0f;
            }
        }
        if constexpr (SPLITS > 0) {
#pragma unroll
            for (int u = 0; u < N; ++u) mx = fmaxf(mx, w[u]);
        }
        const float m_safe = mx == -INFINITY ? 0.0f : mx;
#pragma unroll
        for (int u = 0; u < N; ++u) {
            if (!SPLITS && sp0 + u >= a.splits_total) continue; // uniform (a repeat: 0 x Inf would be NaN)
            const float wu = fast_exp2(w[u] - m_safe);
            lsum += wu * lp[u];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += wu * v[u][i];
        }
    }
    float *dst = a.out + context_row(g, kvh, slot) * g.head_dim + c4;
    const float inv = 1.0f / lsum;
    if (vec_ok && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
        *reinterpret_cast<float4_t *>(dst) = float4_t{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (c4 + i < g.head_dim) dst[i] = acc[i] * inv;
    }
}
__device__ __forceinline__ void merge_rows_body(const DecodeArgs &a, const int kvh, const unsigned block) {
    const unsigned c4n = (unsigned)(a.g.head_dim + 3) >> 2, id = block * 256 + threadIdx.x;
    if (id >= (unsigned)(a.n_queries * a.g.gqa) * c4n) return;
    const int slot = (int)(id / c4n), c4 = (int)(id - (unsigned)slot * c4n) * 4;
    switch (a.splits_total) { // uniform
    case 2: return merge_rows_of<2>(a, kvh, slot, c4);
    case 3: return merge_rows_of<3>(a, kvh, slot, c4);
    case 4: return merge_rows_of<4>(a, kvh, slot, c4);
    default: return merge_rows_of<0>(a, kvh, slot, c4);
    }
}

__global__ __launch_bounds__(256) void merge_rows_kernel(DecodeArgs a) { merge_rows_body(a, blockIdx.y, blockIdx.x); }

static unsigned merge_rows_blocks(const DecodeArgs &a) { // per kv head
    return (unsigned)(((long)a.n_queries * a.g.gqa * ((a.g.head_dim + 3) >> 2) + 255) / 256);
}

hipError_t launch_merge_rows(const DecodeArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(merge_rows_kernel, dim3(merge_rows_blocks(a), (unsigned)a.g.kv_heads), dim3(256), 0, s, a);
    return hipGetLastError();
}

// A ring chunk's last two launches as one: the merge of its partials, and the append of its rows to the
// ring, which nobody reads any more. Workgroups past the merge's append. 3000 tokens in chunks of 512 through
// five rings of q16/kv8/hd256 and 1024 rows: 1777 -> 1752 us.
template <bool F32>
__global__ __launch_bounds__(256) void merge_append_kernel(DecodeArgs a, AppendArgs w, unsigned merge_blocks, unsigned pages) {
    const unsigned kvh = blockIdx.y;
    if (blockIdx.x < merge_blocks) {
        merge_rows_body(a, (int)kvh, blockIdx.x);
    } else {
        const unsigned b = blockIdx.x - merge_blocks, part = b / pages;
        append_tile<F32, 1>(w, (int)(b - part * pages), (int)kvh, (int)part, 256);
    }
}

hipError_t launch_merge_append(const DecodeArgs &a, const AppendArgs &w, hipStream_t s) {
    const AppendGrid r = append_grid(w);
    if (w.n_rows <= 0 || !r.spread) {
        const hipError_t e = launch_merge_rows(a, s);
        return e != hipSuccess ? e : launch_append(w, s);
    }
    const AppendArgs b = append_placed(w);
    const unsigned merge_blocks = merge_rows_blocks(a);
    const dim3 grid(merge_blocks + (unsigned)(r.pages * r.rounds), (unsigned)a.g.kv_heads);
    if (w.g.f32) hipLaunchKernelGGL(merge_append_kernel<true>, grid, dim3(256), 0, s, a, b, merge_blocks, (unsigned)r.pages);
    else hipLaunchKernelGGL(merge_append_kernel<false>, grid, dim3(256), 0, s, a, b, merge_blocks, (unsigned)r.pages);
    return hipGetLastError();
}

// Query slots one workgroup of the kernel covers for a padded head_dim.
int prefill_tile_slots(int P, TileShape shape) {
    if (P > 256) return 64; // four wavefronts, one per SIMD (the accumulators and query halves are 256 registers)
    if (shape == TileShape::two_tiles && P <= 128) return 256;
    return shape == TileShape::halves || (shape == TileShape::quarters && P > 64 && P <= 128) ? 64 : 128;
}

template <int P, int TILES, int SP, int WAVES, int HALVES, bool RING>
static hipError_t launch_tiles_of(const DecodeArgs &a, const ChunkPages &c, dim3 grid, hipStream_t s) {
    constexpr size_t lds = (size_t)TileLds<P, TILES, SP, WAVES, HALVES>::UNITS * sizeof(uint4);
    static_assert(lds <= 160 * 1024, "two steps of pages share the LDS of a compute unit");
    static std::atomic<uint64_t> lds_ok{0}; // per instantiation
    {
        hipError_t e = allow_full_lds(reinterpret_cast<const void *>(&prefill_tile_kernel<P, TILES, SP, WAVES, HALVES, RING>), lds_ok);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((prefill_tile_kernel<P, TILES, SP, WAVES, HALVES, RING>), grid, dim3(WAVES * 64), lds, s, a, c);
    return hipGetLastError();
}
template <int P, int TILES, int SP, int WAVES = 8, int HALVES = 1>
static hipError_t launch_tiles(const DecodeArgs &a, const ChunkPages &c, dim3 grid, hipStream_t s) {
    return c.ring_pages > 0 ? launch_tiles_of<P, TILES, SP, WAVES, HALVES, true>(a, c, grid, s)
                            : launch_tiles_of<P, TILES, SP, WAVES, HALVES, false>(a, c, grid, s);
}

hipError_t launch_prefill_tiles(const DecodeArgs &a, const ChunkPages &c, TileShape shape, hipStream_t s) {
    const int n_slots = a.n_queries * a.g.gqa;
    const int per_wg = prefill_tile_slots(a.g.P, shape);
    const bool two = per_wg == 256, halves = shape == TileShape::halves;
    dim3 grid((unsigned)a.splits, (unsigned)a.g.kv_heads, (unsigned)((n_slots + per_wg - 1) / per_wg));
    switch (a.g.P) {
    case 32:
        if (halves) return launch_tiles<32, 1, 2, 8, 2>(a, c, grid, s);
        return two ? launch_tiles<32, 2, 4>(a, c, grid, s) : launch_tiles<32, 1, 4>(a, c, grid, s);
    case 64:
        if (halves) return launch_tiles<64, 1, 2, 8, 2>(a, c, grid, s);
        return two ? launch_tiles<64, 2, 4>(a, c, grid, s) : launch_tiles<64, 1, 4>(a, c, grid, s);
    case 96:
        if (shape == TileShape::quarters) return launch_tiles<96, 2, 1, 8, 4>(a, c, grid, s);
        if (halves) return launch_tiles<96, 1, 2, 8, 2>(a, c, grid, s);
        return two ? launch_tiles<96, 2, 2>(a, c, grid, s) : launch_tiles<96, 1, 4>(a, c, grid, s);
    case 128:
        if (shape == TileShape::quarters) return launch_tiles<128, 2, 1, 8, 4>(a, c, grid, s);
        if (halves) return launch_tiles<128, 1, 2, 8, 2>(a, c, grid, s);
        return two ? launch_tiles<128, 2, 2>(a, c, grid, s) : launch_tiles<128, 1, 4>(a, c, grid, s);
    case 256:
        if (halves) return launch_tiles<256, 1, 1, 8, 2>(a, c, grid, s);
        return launch_tiles<256, 1, 2>(a, c, grid, s);
    case 512: return launch_tiles<512, 1, 1, 4>(a, c, grid, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace skv

// Device side of the append, shared by its own launch (kernels.hip) and the one that merges a ring chunk's
// partials as well (kernels_prefill.hip).
#pragma once

#include "skv_internal.h"

namespace skv {

__device__ __forceinline__ uint16_t append_bf16_bits(float v) {
    const uint32_t b = __float_as_uint(v);
    return (uint16_t)((b + 0x7fffu + ((b >> 16) & 1u)) >> 16);
}

// ------------------------------------------------------------------------------------
// append: f32 rows -> tiles, bf16 (rounded as above) or f32 (verbatim). One or more workgroups per page of
// positions and kv head; their threads take the tile's 16-byte units as they lie in memory, K units
// (8 or 4 dims of one row) and V units (4 rows of two dims or one), so stores are whole units
// side by side and loads are runs of 64 bytes and more; rows outside the batch leave their K units
// alone, and the V units they share with rows inside are written element by element.
// Stands in for copy_at_f32_to_bf16 (src/decode_resident/kernels.rs:1036-1044).
// Bound by the launch and one round trip up to about a thousand rows, then by memory. Kernel times
// on one MI355X in us, against one thread per (row, 8 or 4 dims) with 64-bit divisions and V stores of an
// element or, in whole groups, one unit: 1 row of 8 x 128 4.1 -> 3.0, 512 rows of 8 x 128 5.0 -> 3.4 (f32 7.6 -> 3.6),
// 32768 rows of 8 x 128 142 -> 92 = 4.4 TB/s (f32 463 -> 121); as calls in a row, 1 row of 2 x 512 f32 2.9 -> 1.9,
// 6 rows of 2 x 256 bf16 4.4 -> 2.2, 130 rows of 8 x 256 f32 5.4 -> 2.4.
// ------------------------------------------------------------------------------------
// UNITS: units of K, and of V, a thread takes; bx, kvh, bz: page of the batch, kv head, which part of the tile
template <bool F32, int UNITS>
__device__ __forceinline__ void append_tile(const AppendArgs &a, const int bx, const int kvh, const int bz, const int threads) {
    typedef __attribute__((ext_vector_type(4))) float f4;
    typedef __attribute__((ext_vector_type(4))) uint32_t w4;
    const Geom g = a.g;
    // The page's place is asked for in front of the rows and looked at behind them, by a vector load, because those come back in
    // order: a scalar one is waited for together with every other, and the rows would be asked for after it.
    int logical = a.first_page + bx;
    if (a.ring_pages > 0 && logical >= a.ring_pages) logical -= a.ring_pages;
    int at = a.table ? logical : 0;
    asm("" : "+v"(at)); // (a vector register)
    const int asked = (a.table ? a.table : reinterpret_cast<const int32_t *>(a.k_src))[at]; // (no table: some valid address)
    const int row0 = bx * 16 - a.first_row; // batch row of the page's first row
    const int r_lo = max(-row0, 0), r_hi = min(16, a.n_rows - row0); // rows of the page in the batch
    const int kv_dim = g.kv_heads * g.head_dim;
    const float *ks = a.k_src + (long)row0 * kv_dim + kvh * g.head_dim;
    const float *vs = a.v_src + (long)row0 * kv_dim + kvh * g.head_dim;
    const int units = g.tile_elems >> 3;
    // K units past head_dim: a layer's pools are zero there from the start, scratch pages are not
    const int k_units = a.table ? ((g.head_dim + (F32 ? 3 : 7)) / (F32 ? 4 : 8)) * 16 : units;
    constexpr int KE = F32 ? 4 : 8; // dims of a K unit
    constexpr int VD = F32 ? 1 : 2; // dims of a V unit

    float kx[UNITS][KE], vx[UNITS][4][VD];
    int kr[UNITS], kd[UNITS], vr[UNITS], vd[UNITS];
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
        const int u = (int)threadIdx.x + (bz * UNITS + i) * threads;
        // unit u of a K tile: row u % 16; dims 8 (u / 16) .., or 16 (u / 64) + 4 (u / 16 % 4) ..
        kr[i] = u & 15;
        kd[i] = (u >> 4) * KE;
        // unit u of a V tile: rows 4 (u / 16 % 4) ..; dims 32 (u / 64) + u % 16 and the one 16 further, or 16 (u / 64) + u % 16
        vr[i] = ((u >> 4) & 3) * 4;
        vd[i] = (u >> 6) * 16 * VD + (u & 15);
        const int row = min(max(kr[i], r_lo), r_hi - 1); // clamped: loads are unconditional, one round trip
        if (a.vec) { // uniform
#pragma unroll
            for (int e = 0; e < KE; e += 4) {
                const f4 x = *reinterpret_cast<const f4 *>(ks + (long)row * kv_dim + min(kd[i] + e, g.head_dim - 4));
#pragma unroll
                for (int t = 0; t < 4; ++t) kx[i][e + t] = x[t];
            }
        } else {
#pragma unroll
            for (int e = 0; e < KE; ++e) kx[i][e] = ks[(long)row * kv_dim + min(kd[i] + e, g.head_dim - 1)];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int vrow = min(max(vr[i] + r, r_lo), r_hi - 1);
#pragma unroll
            for (int d = 0; d < VD; ++d) vx[i][r][d] = vs[(long)vrow * kv_dim + min(vd[i] + 16 * d, g.head_dim - 1)];
        }
    }
    const int page = __builtin_amdgcn_readfirstlane(a.table ? asked : logical);
    const long tile = (long)page * g.page_elems + (long)kvh * g.tile_elems;
    w4 *kt = reinterpret_cast<w4 *>(a.k_pool + tile), *vt = reinterpret_cast<w4 *>(a.v_pool + tile);
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
        const int u = (int)threadIdx.x + (bz * UNITS + i) * threads;
        if (u < k_units && kr[i] >= r_lo && kr[i] < r_hi) {
            w4 w;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if constexpr (F32) {
                    w[t] = kd[i] + t < g.head_dim ? __float_as_uint(kx[i][t]) : 0u;
                } else {
                    const uint32_t lo = kd[i] + 2 * t < g.head_dim ? append_bf16_bits(kx[i][2 * t]) : 0u;
                    const uint32_t hi = kd[i] + 2 * t + 1 < g.head_dim ? append_bf16_bits(kx[i][2 * t + 1]) : 0u;
                    w[t] = lo | (hi << 16);
                }
            }
            kt[u] = w;
        }
        if (u < units && vd[i] < g.head_dim && vr[i] + 3 >= r_lo && vr[i] < r_hi) {
            w4 w;
            if constexpr (F32) {
#pragma unroll
                for (int r = 0; r < 4; ++r) w[r] = __float_as_uint(vx[i][r][0]);
            } else {
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const bool in = vd[i] + 16 * d < g.head_dim;
#pragma unroll
                    for (int r = 0; r < 4; r += 2)
                        w[d * 2 + (r >> 1)] = in ? append_bf16_bits(vx[i][r][d]) | ((uint32_t)append_bf16_bits(vx[i][r + 1][d]) << 16) : 0u;
                }
            }
            if (vr[i] >= r_lo && vr[i] + 4 <= r_hi) {
                vt[u] = w;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (vr[i] + r < r_lo || vr[i] + r >= r_hi) continue;
                    if constexpr (F32) {
                        reinterpret_cast<uint32_t *>(vt + u)[r] = w[r];
                    } else {
                        uint16_t *dst = reinterpret_cast<uint16_t *>(vt + u);
                        dst[r] = (uint16_t)(w[r >> 1] >> ((r & 1) * 16));
                        dst[4 + r] = (uint16_t)(w[2 + (r >> 1)] >> ((r & 1) * 16));
                    }
                }
            }
        }
    }
}

// How a launch of 256-thread workgroups divides a batch: pages x kv heads x parts of a tile. A tile of more
// than 256 units is shared by workgroups of 256 units each while those are at most 4096, else one workgroup
// takes it whole, several units a thread: shared / whole in us, 1 row of 2 x 512 f32 1.9/4.2, 512 rows of
// 2 x 256 bf16 2.4/3.0, of 2 x 512 2.8/4.4, of 8 x 256 3.4/3.9 (f32 3.7/4.3), 2048 rows of 8 x 256 7.4/7.7 (f32, 4128
// workgroups, 10.2/9.4).
struct AppendGrid {
    long pages;
    int rounds;  // workgroups' worth of units in a tile
    bool spread; // one workgroup each
};
inline AppendGrid append_grid(const AppendArgs &a) {
    AppendGrid r;
    r.pages = (a.first_pos + a.n_rows + 15) / 16 - a.first_pos / 16;
    r.rounds = ((a.g.tile_elems >> 3) + 255) / 256;
    r.spread = r.pages * a.g.kv_heads * r.rounds <= 4096;
    return r;
}
// What the launch wants to know of a: 16-byte loads of K, and the places of its pages
inline AppendArgs append_placed(const AppendArgs &a) {
    AppendArgs b = a;
    b.vec = ((uintptr_t)a.k_src & 15) == 0 && (a.g.head_dim & 3) == 0;
    b.first_page = (int)(slot_of(a.first_pos / 16 * 16, a.g.ring_rows) / 16);
    b.first_row = (int)(a.first_pos % 16);
    b.ring_pages = a.g.ring_rows / 16;
    return b;
}

} // namespace skv

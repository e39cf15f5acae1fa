// Device side of the fused pre-KV step (per-head RMSNorm and rotation of the group's queries and of
// the new k row), shared by the decode kernels of both elements.
#pragma once

#include "skv_internal.h"

namespace skv {

// Entry `i` of a block table, the same in every lane, through the scalar unit: counted apart from the
// vector loads in flight. The compiler takes the vector unit where it cannot prove the index uniform
// (in the pre-KV kernels), and then waits for every load issued before: SAID says that it is.
template <bool SAID>
__device__ __forceinline__ int table_entry(const int32_t *table, int i) {
    typedef const __attribute__((address_space(4))) int32_t *const_i32_ptr;
    return reinterpret_cast<const_i32_ptr>(reinterpret_cast<uintptr_t>(table))[SAID ? __builtin_amdgcn_readfirstlane(i) : i];
}

// Used by one workgroup of a decode launch while its first page is in flight:
//   load()   asks for the raw rows, the weights and the rotation (before the first page);
//   stage()  puts them into LDS with the squares; barrier;
//   scales() lane r of the workgroup sums the squares of row r in index order; barrier;
//   each()   hands every finished unit of four dims to the caller, who stores it where its products
//            read it.
// The arithmetic and its order are those of rms_norm_rope_heads_at (src/decoder/attention_ops.rs:682-777),
// so the finished rows, and the k row the launch stores, equal the CPU path's bit for bit.
// What bounds it is the chain load, LDS, ordered sum, LDS: nothing of it can overlap the products. So
// rows pass through LDS in 16-byte units, the sum's reads are a round ahead of its adds, and no row
// is written back between the rotation and the operand layout. Two tokens through 36 bf16 layers of
// q32/kv8/hd128 over 2048 rows: 705 -> 616 us of GPU time, with the first page's table entry read through the
// scalar unit (the page's requests had waited for the queries) and its V asked for behind the sums.
template <int P, int THREADS>
struct PreKvStage {
    typedef __attribute__((ext_vector_type(4))) float f4;
    static constexpr int ROWS = 17; // 16 query slots and the new k row
    static constexpr int P4 = P / 4;
    static constexpr int RS = P + 4; // row stride: 16-byte aligned, lanes on different rows hit different banks
    static constexpr int U = (16 * P4 + THREADS - 1) / THREADS;
    static constexpr int NE = (P + THREADS - 1) / THREADS;
    static constexpr size_t LDS_FLOATS = (size_t)2 * ROWS * RS + 3 * P + ROWS + 3;

    f4 q[U];
    float wq[NE], wk[NE], rot[NE];

    __device__ __forceinline__ static float *sq(float *lds) { return lds + ROWS * RS; }
    __device__ __forceinline__ static float *weights(float *lds) { return lds + 2 * ROWS * RS; } // q's [P], k's [P]
    __device__ __forceinline__ static float *rotation(float *lds) { return weights(lds) + 2 * P; } // [P]: (cos, sin)
    __device__ __forceinline__ static float *inv(float *lds) { return weights(lds) + 3 * P; }      // [ROWS]

    __device__ __forceinline__ void load(const DecodeArgs &a, int kvh, int rows, int q_stride, int tid) {
        const int hd = a.g.head_dim;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = tid + u * THREADS;
            const int r = e / P4, c = (e % P4) * 4;
            q[u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
            if (r < rows) {
                const float *row = a.q + (long)(kvh * a.g.gqa + r) * q_stride;
                if (a.q_vec) {
                    q[u] = *reinterpret_cast<const f4 *>(row + min(c, hd - 4));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[u][i] = row[min(c + i, hd - 1)];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < NE; ++u) {
            const int d = tid + u * THREADS;
            wq[u] = (a.q_norm_w && d < hd) ? a.q_norm_w[d] : 1.0f;
            wk[u] = (a.k_norm_w && d < hd) ? a.k_norm_w[d] : 1.0f;
            rot[u] = (a.rope && d < a.rope_dims) ? a.rope[d] : 0.0f;
        }
    }

    // k_rows: elements tid, tid + THREADS, .. of the raw new row (zeros where the workgroup appends none)
    __device__ __forceinline__ void stage(float *lds, const DecodeArgs &a, int rows, const float (&k_rows)[NE], int tid) {
#pragma clang fp contract(off)
        const int hd = a.g.head_dim;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = tid + u * THREADS;
            const int r = e / P4, c = (e % P4) * 4;
            if (r < rows) {
                f4 x = q[u];
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = c + i < hd ? x[i] : 0.0f;
                *reinterpret_cast<f4 *>(lds + r * RS + c) = x;
                *reinterpret_cast<f4 *>(sq(lds) + r * RS + c) = x * x;
            }
        }
#pragma unroll
        for (int u = 0; u < NE; ++u) {
            const int d = tid + u * THREADS;
            if (d < P) {
                lds[rows * RS + d] = k_rows[u];
                sq(lds)[rows * RS + d] = k_rows[u] * k_rows[u];
                weights(lds)[d] = wq[u];
                weights(lds)[P + d] = wk[u];
                rotation(lds)[d] = rot[u];
            }
        }
    }

    __device__ __forceinline__ static void scales(float *lds, const DecodeArgs &a, int rows, int n_rows, int tid) {
        if (tid >= n_rows) return;
        const bool has_norm = tid == rows ? a.k_norm_w != nullptr : a.q_norm_w != nullptr;
        inv(lds)[tid] = has_norm ? head_inv_rms_sq<P>(sq(lds) + tid * RS, a.g.head_dim, a.eps) : 1.0f;
    }

    // f(r, c4, v): v = dims 4 c4 .. +3 of finished row r (row `rows` is the k row), zeros past head_dim
    template <typename F>
    __device__ __forceinline__ static void each(float *lds, const DecodeArgs &a, int rows, int n_rows, int tid, F &&f) {
#pragma clang fp contract(off)
        const int hd = a.g.head_dim, half = a.rope_dims >> 1;
        // whole units everywhere: the rotation's partners are a unit of the same row, or this one's own dims
        const bool units = (hd & 3) == 0 && (!a.rope || (a.rope_dims & (a.rope_style == 1 ? 3 : 7)) == 0);
        for (int e = tid; e < n_rows * P4; e += THREADS) {
            const int r = e / P4, c4 = e % P4, c = c4 * 4;
            const float *row = lds + r * RS;
            const float *w = weights(lds) + (r == rows ? P : 0); // ones where there is no weight
            const float *rp = rotation(lds);
            const float iv = inv(lds)[r];
            f4 n = f4{0.0f, 0.0f, 0.0f, 0.0f};
            if (units) {
                const f4 x = *reinterpret_cast<const f4 *>(row + c), wx = *reinterpret_cast<const f4 *>(w + c);
                if (a.rope && c < a.rope_dims) {
                    if (a.rope_style == 1) {
                        n = norm_rope_unit(x, x, wx, wx, *reinterpret_cast<const f4 *>(rp + c), x, iv, 1, true);
                    } else {
                        const bool is_first = c < half;
                        const int oc = is_first ? c + half : c - half, b = is_first ? c : oc;
                        n = norm_rope_unit(x, *reinterpret_cast<const f4 *>(row + oc), wx, *reinterpret_cast<const f4 *>(w + oc),
                                           *reinterpret_cast<const f4 *>(rp + 2 * b),
                                           *reinterpret_cast<const f4 *>(rp + 2 * b + 4), iv, 0, is_first);
                    }
                } else {
                    n = x * iv;
                    n = n * wx;
                }
                if (c >= hd) n = f4{0.0f, 0.0f, 0.0f, 0.0f};
            } else {
                const float *wn = (r == rows ? a.k_norm_w : a.q_norm_w) ? w : nullptr;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (c + i < hd) n[i] = norm_rope_elem(row, c + i, iv, wn, a.rope ? rp : nullptr, a.rope_dims, a.rope_style);
            }
            f(r, c4, n);
        }
    }
};

} // namespace skv

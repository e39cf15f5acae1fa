// Device side of ChunkPages (skv_internal.h), shared by the prefill kernels of both elements.
#pragma once

#include "skv_internal.h"

namespace skv {

// Entry e of the launch's page list: where its tiles lie (of the workgroup's kv head, in 16-byte
// units from its pool's start), which position its first row has, and the first and last
// position whose rows it may speak for. On full layers entry e is logical page e.
template <bool RING>
__device__ __forceinline__ uint32_t entry_place(const DecodeArgs &a, const ChunkPages &c, int e) { // physical page
    if constexpr (RING) {
        int at = c.start + min(e, c.n_old - 1);
        if (at >= c.ring_pages) at -= c.ring_pages;
        const int page = a.table[max(at, 0)];
        return (uint32_t)(e < c.n_old ? page : e - c.n_old);
    } else {
        return (uint32_t)a.table[e];
    }
}
__device__ __forceinline__ uint32_t place_tile(const DecodeArgs &a, uint32_t place, int kvh) {
    return place * (uint32_t)(a.g.page_elems >> 3) + (uint32_t)kvh * (uint32_t)(a.g.tile_elems >> 3);
}
template <bool RING>
__device__ __forceinline__ uint32_t entry_tile(const DecodeArgs &a, const ChunkPages &c, int e, int kvh) {
    return place_tile(a, entry_place<RING>(a, c, e), kvh);
}
template <bool RING>
__device__ __forceinline__ int entry_pos(const ChunkPages &c, int e) {
    if constexpr (!RING) return e * 16;
    return e < c.n_old ? c.first_pos + e * 16 : c.new_first + (e - c.n_old) * 16;
}
template <bool RING>
__device__ __forceinline__ int entry_lo(const ChunkPages &c, int e) {
    return !RING || e < c.n_old ? INT32_MIN : c.new_pos0;
}
template <bool RING>
__device__ __forceinline__ int entry_hi(const ChunkPages &c, int e) {
    return !RING || e >= c.n_old ? INT32_MAX : c.new_pos0 - 1;
}
// The entries [e0, e1) of [first, last) all of whose rows lie in [lo, hi] and are the entry's to
// speak for, as two ranges: old entries, new ones.
struct Inner {
    int o0, o1, n0, n1;
};
template <bool RING>
__device__ __forceinline__ Inner inner_entries(const ChunkPages &c, int first, int last, int lo, int hi) {
    Inner r;
    if constexpr (!RING) {
        r.o0 = max(first, (lo + 15) >> 4);
        r.o1 = min(last, (hi - 15 >= 0 ? (hi - 15) >> 4 : -1) + 1);
        r.n0 = r.n1 = 0;
    } else {
        r.o0 = max(first, (lo - c.first_pos + 15) >> 4);
        r.o1 = min(min(last, c.n_old), ((min(hi, c.new_pos0 - 1) - 15 - c.first_pos) >> 4) + 1);
        r.n0 = max(max(first, c.n_old), c.n_old + ((max(lo, c.new_pos0) - c.new_first + 15) >> 4));
        r.n1 = min(last, c.n_old + ((hi - 15 - c.new_first) >> 4) + 1);
    }
    return r;
}

} // namespace skv

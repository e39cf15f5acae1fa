// Copies straight from memory to LDS, shared by the prefill kernels of both elements.
#pragma once

#include "skv_internal.h"

namespace skv {

// 64 x 16 bytes straight from memory to LDS, lane l's to lds + 16 l (`lds` the same in every lane), no
// register in between. In assembly because the compiler, which cannot tell the parts of a
// kernel's buffers apart, would make every LDS read wait for a copy it knows of; the kernel
// waits for them itself (copies_landed, copies_left) in front of the barrier that hands the buffer over.
// `kib`: a constant, that many KiB further at both ends (an immediate of the instruction).
__device__ __forceinline__ void copy_to_lds(const void *base, uint32_t lane_offset, uint32_t lds, int kib = 0) {
    // (both are the same in every lane: said so, whatever the compiler can prove)
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint64_t from = ((uint64_t)hi << 32) | lo;
    const uint32_t to = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
    switch (kib) {
    case 0: asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(lane_offset), "s"(from) : "m0"); break;
    case 1: asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024" ::"s"(to), "v"(lane_offset), "s"(from) : "m0"); break;
    case 2: asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:2048" ::"s"(to), "v"(lane_offset), "s"(from) : "m0"); break;
    default: asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072" ::"s"(to), "v"(lane_offset), "s"(from) : "m0"); break;
    }
}
__device__ __forceinline__ void copies_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// all but the wavefront's last N copies have landed
template <int N>
__device__ __forceinline__ void copies_left() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

} // namespace skv

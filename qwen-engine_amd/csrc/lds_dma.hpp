// Loads from memory straight into LDS (global_load_lds), written out: the
// compiler cannot tell which buffer a load in flight fills and would wait for
// it at the next read of LDS.  The caller holds the waits (s_waitcnt vmcnt and a
// barrier) between a load and the reads of what it fills, and before the block
// ends.  dst is the wave-uniform LDS byte address of lane 0's piece; lane l's goes
// to dst + l * 16 (x4) or dst + l * 4 (dword; ushort: two bytes, zero-extended).
//
// Every statement names m0 as written.  clang warns that the register is a
// reserved one; the passes that merge or hoist settings of m0 do look at the list.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qe {

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load_x4(uint32_t dst, const void* base, uint32_t lane_offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 ::"s"(dst), "v"(lane_offset), "s"(base) : "m0", "memory");
}
__device__ __forceinline__ void lds_load_x4(uint32_t dst, const void* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "m0", "memory");
}
__device__ __forceinline__ void lds_load_dword(uint32_t dst, const void* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src) : "m0", "memory");
}
__device__ __forceinline__ void lds_load_ushort(uint32_t dst, const void* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, off" ::"s"(dst), "v"(src) : "m0", "memory");
}
#pragma clang diagnostic pop

}  // namespace qe

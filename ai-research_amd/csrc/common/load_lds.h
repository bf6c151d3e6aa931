// load_lds.h -- direct loads from memory to LDS: 16 bytes per lane from the
// lane's address to LDS byte lds + 16 * lane (lds uniform).  They complete in
// order with the wave's other loads and are waited for with vmcnt; the compiler
// does not know of them, so the kernels write the waits out.  (It notes that m0 is
// a reserved register: its own uses set m0 just ahead, and the clobber keeps them
// from sharing a value across these.)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

__device__ __forceinline__ void load_lds16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
               : "memory", "m0");
}
// from base + off, base uniform
__device__ __forceinline__ void load_lds16(uint32_t off, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}

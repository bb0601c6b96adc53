// Loads from memory straight to LDS, and the waits that go with them (gfx950). They are asm
// because the compiler would wait for every load in flight before any LDS read; they write
// no vector register. `wait_loads` and a barrier come before the data are read.
#pragma once

#include "common.h"

namespace amd_ops {
namespace fa {

// LDS address of shared memory: what the loads below add their lanes' 16 bytes to. Never a
// bare offset, which would take for granted that nothing else lies in the kernel's LDS.
__device__ __forceinline__ unsigned lds_address(const void* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// 16 bytes a lane, 1024 consecutive ones of LDS a wave: from `base` + the lane's `off`
__device__ __forceinline__ void load_lds16(unsigned lds, const void* base, unsigned off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
// the same of data that is read once: it leaves no trace in the caches
__device__ __forceinline__ void load_lds16_once(unsigned lds, const void* base, unsigned off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
               :: "s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
// the same from an address of the lane's own
__device__ __forceinline__ void load_lds16(unsigned lds, const void* mine) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds), "v"(mine) : "memory", "m0");
}

// waits until at most LATER of the wave's loads, the last ones issued, are in flight
template <int LATER = 0>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LATER) : "memory");
}

// barrier behind which every wave's LDS reads so far are complete
__device__ __forceinline__ void barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace fa
}  // namespace amd_ops

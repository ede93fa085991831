// Memory straight into LDS: what the kernels that keep a ring of blocks there share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// One load of 16 bytes per lane from global memory straight into LDS, written as the instruction itself. Through the
// compiler's builtin the compiler knows of a load into LDS that is on its way, and from then on it waits for all
// outstanding loads and LDS reads before every use of either (it cannot tell which of them that load might be): the
// kernels write the waits by hand instead, as their pipelines need them. `lds` is the byte address in LDS of the wave's 1 KB
// (m0 holds it, lane l's 16 bytes land at lds + 16 l).
__device__ __forceinline__ void load_to_lds_16(const void* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds_16(const void* address, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(address), "s"(lds) : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_loads() {  // until at most N of the wave's loads are in flight
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Rows of 128 bytes, eight to a load: the piece of row r in slot s is s ^ ring_swz(r), so that 16 lanes that read one piece of
// 16 rows cover the 64 banks once, and 8 lanes of 8 rows half of them. A lane's place in LDS is fixed by its number, so the
// swizzle is applied on the global side.
__device__ __forceinline__ int ring_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

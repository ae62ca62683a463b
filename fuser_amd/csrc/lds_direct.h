// LDS-direct loads of gfx950: global memory -> LDS without a register in between.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvf {
namespace {

// Lane L's 16 (4) bytes at base + voff go to lds_byte_addr + OFFSET + 16 * L (4 * L); lds_byte_addr and base are
// wave-uniform.  Issued from inline assembly: the compiler neither waits for the load nor orders LDS reads against it, the
// kernels do that with explicit s_waitcnt vmcnt(n).
// The LDS address is passed in m0, and a load that uses m0 needs one wait state after a scalar instruction has written it,
// or it may still see the last load's address.  The compiler cannot insert the state inside an asm string, so it is here.
// STREAM: non-temporal, for data that the last-level cache cannot hold anyway.
#define NVF_LDS_DIRECT(load)                                                                                             \
  if constexpr (OFFSET == 0)                                                                                             \
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" load ::"s"(lds_byte_addr), "v"(voff), "s"(base) : "memory", "m0");    \
  else                                                                                                                   \
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\t" load ::"s"(lds_byte_addr), "v"(voff), "s"(base), "i"(OFFSET)      \
                 : "memory", "m0", "scc")

template <int OFFSET = 0, bool STREAM = false>
__device__ __forceinline__ void lds_dma16(uint32_t lds_byte_addr, const uint8_t* base, uint32_t voff) {
  if constexpr (STREAM) {
    NVF_LDS_DIRECT("global_load_lds_dwordx4 %1, %2 nt");
  } else {
    NVF_LDS_DIRECT("global_load_lds_dwordx4 %1, %2");
  }
}

template <int OFFSET = 0>
__device__ __forceinline__ void lds_dma4(uint32_t lds_byte_addr, const uint8_t* base, uint32_t voff) {
  NVF_LDS_DIRECT("global_load_lds_dword %1, %2");
}
#undef NVF_LDS_DIRECT

}  // namespace
}  // namespace nvf

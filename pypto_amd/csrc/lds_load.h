// Direct global -> LDS requests of the GEMM kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace pto_hip {

// One direct request: 16 bytes per lane from `src` to the KB of LDS at lds_w + OFF (wave-uniform).
// The instruction is written out: told that a load writes LDS, the compiler waits for every such
// load in flight before each later LDS read, whatever buffer that read addresses.  It does not look into
// the string for hazards either: the ISA asks for one wait state between a scalar write of m0 and a load that
// takes its LDS address from it, hence s_nop.
template <int OFF>
__device__ __forceinline__ void to_lds(const void* src, uint32_t lds_w) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is named as clobbered on purpose
  asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_w), "n"(OFF)
               : "memory", "m0", "scc");
#pragma clang diagnostic pop
}

// ... from sbase + voff, the base wave-uniform: no 64-bit address per lane and request.
template <int OFF>
__device__ __forceinline__ void to_lds(uint32_t voff, const void* sbase, uint32_t lds_w) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_w), "n"(OFF)
               : "memory", "m0", "scc");
#pragma clang diagnostic pop
}

}  // namespace pto_hip

// Instantiations of the products of a small call: fp16 operands.
#include "narrow_gemm.h"

namespace pto_hip {
int narrow_dual_fp16(const gemm::GemmParams& p, int tile, hipStream_t st) {
  return gemm::launch_narrow<false, true, _Float16>(p, tile, st);
}
int narrow_single_fp16(const gemm::GemmParams& p, int tile, int out_dtype, hipStream_t st) {
  return out_dtype == PTO_HIP_FP32 ? gemm::launch_narrow<false, false, float>(p, tile, st)
                                   : gemm::launch_narrow<false, false, _Float16>(p, tile, st);
}
}  // namespace pto_hip

// Instantiations of the tiled GEMM: fp16 weights, one operand (projections, the down pass).
#include "gemm.h"

namespace pto_hip {
int gemm_launch_w16_single_fp16(const gemm::GemmParams& p, int out_dtype, hipStream_t st) {
  return gemm::launch_by_out<false, false, false>(p, out_dtype, st);
}
}  // namespace pto_hip

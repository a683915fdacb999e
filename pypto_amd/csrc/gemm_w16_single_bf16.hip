// Instantiations of the tiled GEMM: bf16 weights, one operand (projections, the down pass).
#include "gemm.h"

namespace pto_hip {
int gemm_launch_w16_single_bf16(const gemm::GemmParams& p, int out_dtype, hipStream_t st) {
  return gemm::launch_by_out<false, true, false>(p, out_dtype, st);
}
}  // namespace pto_hip

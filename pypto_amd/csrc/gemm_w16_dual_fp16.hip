// Instantiations of the tiled GEMM: fp16 weights, gate/up pair with SwiGLU.
#include "gemm.h"

namespace pto_hip {
int gemm_launch_w16_dual_fp16(const gemm::GemmParams& p, int out_dtype, hipStream_t st) {
  return gemm::launch_by_out<true, false, false>(p, out_dtype, st);
}
}  // namespace pto_hip

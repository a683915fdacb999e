// Instantiations of the tiled GEMM: int8 weight codes, one operand.
#include "gemm.h"

namespace pto_hip {
int gemm_launch_w8_single(const gemm::GemmParams& p, int dtype, int out_dtype, hipStream_t st) {
  return dtype == PTO_HIP_BF16 ? gemm::launch_by_out<false, true, true>(p, out_dtype, st)
                               : gemm::launch_by_out<false, false, true>(p, out_dtype, st);
}
}  // namespace pto_hip

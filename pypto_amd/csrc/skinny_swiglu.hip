// Skinny projections that make their activations themselves: SwiGLU of the pair in front.
#include "skinny.h"

namespace pto_hip {
int skinny_swiglu_launch(const skinny::GemvParams& p, bool bf16, bool w16, bool wide, int wgs, size_t smem, hipStream_t st) {
  return skinny::launch_fused_source<skinny::kSwiglu>(p, bf16, w16, wide, wgs, smem, st);
}
}  // namespace pto_hip

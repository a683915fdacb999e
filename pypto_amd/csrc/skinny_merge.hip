// Skinny projections that make their activations themselves: attention partials merged.
#include "skinny.h"

namespace pto_hip {
int skinny_merge_launch(const skinny::GemvParams& p, bool bf16, bool w16, bool wide, int wgs, size_t smem, hipStream_t st) {
  return p.src.head_dim == 256 ? skinny::launch_fused_source<skinny::kMerge256>(p, bf16, w16, wide, wgs, smem, st)
                               : skinny::launch_fused_source<skinny::kMerge128>(p, bf16, w16, wide, wgs, smem, st);
}
}  // namespace pto_hip

// Instantiations of the weight-streaming projections of some tens of rows: 16-bit weights.
#include "stream_rows.h"

namespace pto_hip {
int stream_rows_w16(const stream::StreamParams& p, bool bf16, hipStream_t st) {
  return bf16 ? stream::launch_w16<true>(p, st) : stream::launch_w16<false>(p, st);
}
}  // namespace pto_hip

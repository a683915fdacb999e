// Instantiations of the weight-streaming projections of some tens of rows: int8 codes.
#include "stream_rows.h"

namespace pto_hip {
int stream_rows_w8(const stream::StreamParams& p, bool bf16, hipStream_t st) {
  return bf16 ? stream::launch_w8<true>(p, st) : stream::launch_w8<false>(p, st);
}
}  // namespace pto_hip

// Which projections of some tens of rows stream their weights (stream_rows.h), and their launch.
#include "launch_choice.h"
#include "stream_rows.h"

#include <algorithm>

namespace pto_hip {
int stream_rows_w8(const stream::StreamParams& p, bool bf16, hipStream_t st);
int stream_rows_w16(const stream::StreamParams& p, bool bf16, hipStream_t st);

int stream_rows_for(int64_t m, int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16, hipStream_t st) {
  const int mats = wq1 ? 2 : 1;
  if (ctx().gemm_stream == 0 || ctx().gemm_variant != 0 || ctx().gemm_splits != 0 || ctx().gemm_quad_rows != 0) return 0;
  if (w16 && ctx().gemm_narrow > 0) return 0;  // a tile of the small-call form is asked for
  if (k % 8 != 0 || k < 32 || n % 8 != 0 || (n + 127) / 128 * mats > ctx().num_cu || ((uintptr_t)wq0 | (uintptr_t)wq1) % 16 != 0) return 0;
  if (m <= kW8MaxM || m > kStreamRowsMax || (ctx().gemm_stream == 1 && !stream_rows_ahead(m, k, n, mats == 2, w16, ctx().num_cu))) return 0;
  void* area = nullptr;
  if (gemm_slabs((size_t)stream_splits(k, n, mats == 2, ctx().num_cu) * mats * m * n * sizeof(float), st, &area) || !area) return 0;
  return (int)((m + 15) / 16 * 16);
}

int stream_partials(const void* x, int x_rows, const void* wq0, const void* wq1, int64_t m, int64_t k, int64_t n, int x_dtype,
                    hipStream_t st, W8Partials* out, bool w16) {
  stream::StreamParams p{};
  p.x = reinterpret_cast<const uint16_t*>(x);
  p.w[0] = wq0;
  p.w[1] = wq1;
  p.m = (int)m;
  p.k = (int)k;
  p.n = (int)n;
  p.x_rows = x_rows;
  p.mats = wq1 ? 2 : 1;
  p.slabs = (int)((n + 127) / 128);
  p.ks = (int)((k + 31) / 32);
  p.splits = stream_splits(k, n, p.mats == 2, ctx().num_cu);
  void* area = nullptr;
  int rc = gemm_slabs((size_t)p.splits * p.mats * m * n * sizeof(float), st, &area);
  if (rc) return rc;
  PTO_CHECK_ARG(area != nullptr, "stream_partials: no room for the slabs");
  p.part = reinterpret_cast<float*>(area);
  rc = w16 ? stream_rows_w16(p, x_dtype == PTO_HIP_BF16, st) : stream_rows_w8(p, x_dtype == PTO_HIP_BF16, st);
  if (rc) return rc;
  *out = W8Partials{};
  out->part[0] = p.part;
  out->part[1] = wq1 ? p.part + (size_t)p.splits * m * n : nullptr;
  out->splits = p.splits;
  out->slab_stride = m * n;
  return PTO_HIP_OK;
}

}  // namespace pto_hip

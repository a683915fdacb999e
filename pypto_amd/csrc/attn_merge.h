// Merge of one output row's attention partials by a wavefront: the merge launch and the o-projection that merges for itself.
#pragma once

#include <hip/hip_runtime.h>

namespace pto_hip {
namespace attn {

constexpr float kMinMax = -1e30f;  // clamp of the running maximum (04_paged_attention.py:521)

// Merge of the per-partition (m, l, o): the online-update algebra of
// examples/models/04_paged_attention.py:186-215 applied across partitions, then o / l.
// One wavefront per output row; lane i gets channels i, i + 64, ...  n_part: slots of a row, np: those in use.  What bounds it is the chain of memory round trips: one up to 8 partitions, above that one for
// the context length, one for the first BATCH partials and less than one for every BATCH more.  BATCH 0: launches of up to kReduceFast partitions, a kernel
// of its own: beside the other path's two batches of partials (16 then) it held 132 registers instead of 50 (head_dim 256: 226 instead of 64), two or three
// wavefronts per SIMD instead of eight.  Attention call of 128 sequences, 32 heads on one KV head, one kernel for both -> two, us: 16-bit
// cache of 1024 tokens 30.3 -> 29.0, of 64 to 4096 42.7 -> 38.0, e4m3 27.9 -> 25.5 and 45.2 -> 36.1.
constexpr int kReduceFast = 8;  // most partitions of the path without a loop
template <int D, int BATCH>
__device__ __forceinline__ void merge_row(const float* ml, const float* po, int n_part, int np, int lane, float (&y)[D / 64]) {
  if constexpr (BATCH == 0) {
    // Few partitions: every slot the row could use is fetched at once, before the context length
    // is known, so the launch is one memory round trip instead of three; slots past np (never
    // written, or stale) are dropped by select, not by a zero weight.
    float pm[kReduceFast], pl[kReduceFast], pv[kReduceFast][D / 64];
#pragma unroll
    for (int u = 0; u < kReduceFast; ++u) {
      const int i = min(u, n_part - 1);
      pm[u] = ml[2 * i];
      pl[u] = ml[2 * i + 1];
#pragma unroll
      for (int k = 0; k < D / 64; ++k) pv[u][k] = po[(size_t)i * D + k * 64 + lane];
    }
    float m = kMinMax;
#pragma unroll
    for (int u = 0; u < kReduceFast; ++u) m = u < np ? fmaxf(m, pm[u]) : m;
    float l = 0.f, o[D / 64];
#pragma unroll
    for (int k = 0; k < D / 64; ++k) o[k] = 0.f;
#pragma unroll
    for (int u = 0; u < kReduceFast; ++u) {
      const float wgt = __builtin_amdgcn_exp2f(pm[u] - m);
      if (u < np) {
        l += wgt * pl[u];
#pragma unroll
        for (int k = 0; k < D / 64; ++k) o[k] += wgt * pv[u][k];
      }
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int k = 0; k < D / 64; ++k) y[k] = o[k] * inv;
    return;
  }
  // Lane i holds (m, l) of partitions i, i + 64, ...  Every batch of partials is requested before the one in front of it is summed.
  // Slots past the row's own partitions repeat its last one, a line that is asked for anyway, and are dropped by select: all slots asked for before
  // the length is known cost the other rows' bandwidth (100 sequences of 16 to 2500 tokens, 32 heads on one KV head at head_dim 256, 50.5 -> 49.3 us).
  constexpr int kBatch = BATCH == 0 ? 1 : BATCH;  // (not instantiated past the return above)
  const int last = max(np - 1, 0);
  float pv[2][kBatch][D / 64];
  auto fetch = [&](int set, int first) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int k = 0; k < D / 64; ++k) pv[set][u][k] = po[(size_t)min(first + u, last) * D + k * 64 + lane];
  };
  float2 own = *reinterpret_cast<const float2*>(ml + 2 * min(lane, last));
  fetch(0, 0);
  float m = lane < np ? own.x : kMinMax;
  for (int i = lane + 64; i < np; i += 64) m = fmaxf(m, ml[2 * i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  float l = 0.f, o[D / 64];
#pragma unroll
  for (int k = 0; k < D / 64; ++k) o[k] = 0.f;
  for (int base = 0; base < np; base += 64) {
    if (base > 0) own = *reinterpret_cast<const float2*>(ml + 2 * min(base + lane, last));
    const float wgt = base + lane < np ? __builtin_amdgcn_exp2f(own.x - m) : 0.f;
    l += base + lane < np ? wgt * own.y : 0.f;
    auto add = [&](int set, int first) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wgt), (first + u) & 63));
#pragma unroll
        for (int k = 0; k < D / 64; ++k) o[k] = first + u < np ? o[k] + w * pv[set][u][k] : o[k];
      }
    };
    for (int first = base; first < min(base + 64, np); first += 2 * kBatch) {
      if (first + kBatch < np) fetch(1, first + kBatch);
      add(0, first);
      if (first + 2 * kBatch < np) fetch(0, first + 2 * kBatch);
      if (first + kBatch < np) add(1, first + kBatch);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int k = 0; k < D / 64; ++k) y[k] = o[k] * inv;
}

}  // namespace attn
}  // namespace pto_hip

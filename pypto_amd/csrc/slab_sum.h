// Sum of a projection's partial slabs by its consumers (finish kernels, RoPE).
#pragma once

#include <hip/hip_runtime.h>

namespace pto_hip {

// V (float or a vector of floats) from an address that need only be a float's: callers' tensors may start at any float,
// and a template argument does not carry a lower alignment of a vector type.
template <typename V>
__device__ __forceinline__ V load_floats(const float* src) {
  V v;
  __builtin_memcpy(&v, src, sizeof(V));
  return v;
}

template <int N, int K, typename V>
__device__ __forceinline__ void add_slab_batch(const float* const (&src)[K], size_t stride, V (&sum)[K]) {
  V t[K][N];
#pragma unroll
  for (int s = 0; s < N; ++s)
#pragma unroll
    for (int k = 0; k < K; ++k) t[k][s] = load_floats<V>(src[k] + s * stride);
#pragma unroll
  for (int s = 0; s < N; ++s)
#pragma unroll
    for (int k = 0; k < K; ++k) sum[k] += t[k][s];
}

// sum[k] += src[k][0] + src[k][stride] + ... (count of them), added in order; stride in floats.
// These kernels are a chain of memory round trips (the slabs come from other XCDs' workgroups): up to
// eight slabs of every source are requested at once, whatever the count, where a remainder loop makes one trip
// per slab.  Decoder layer of one sequence, int8 weights (2 to 8 slabs a channel): batches of four and a serial
// remainder, the two channels of a rotated pair and the gate and up sums one after the other 74.5 us, so 73.1.
template <int K, typename V>
__device__ __forceinline__ void add_slabs(const float* const (&first)[K], int count, size_t stride, V (&sum)[K]) {
  const float* src[K];
#pragma unroll
  for (int k = 0; k < K; ++k) src[k] = first[k];
  for (int left = count; left > 0; left -= 8) {
    switch (left) {
      case 1: add_slab_batch<1>(src, stride, sum); break;
      case 2: add_slab_batch<2>(src, stride, sum); break;
      case 3: add_slab_batch<3>(src, stride, sum); break;
      case 4: add_slab_batch<4>(src, stride, sum); break;
      case 5: add_slab_batch<5>(src, stride, sum); break;
      case 6: add_slab_batch<6>(src, stride, sum); break;
      case 7: add_slab_batch<7>(src, stride, sum); break;
      default: add_slab_batch<8>(src, stride, sum); break;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) src[k] += 8 * stride;
  }
}

}  // namespace pto_hip

// e4m3 products of few rows, or of small matrices, in one launch each: c[M, N] = A8[M, K] @ B8[N, K]^T with row and channel scales, or
// SiLU of one such product times another.
//
// Such a product is bound by its chain: the tiled GEMM (ffn_fp8.hip) has 128 rows x 256 channels a workgroup and walks k with a barrier
// a stage; a few rows leave most CUs idle, or k is split and a second launch sums the slabs.  Here a tile is 16 to 64 rows x 16 or 32
// channels, the workgroup's wavefronts split k among themselves (no slabs, no second launch), and both operands, which are
// k-contiguous, go straight from memory to MFMA registers: the lane of row c and group kg takes the 32 codes from k = 32 kg of a step of 128, of activations
// and weights alike.  Every tile reads its operands for itself, which is why it stops paying at a few hundred rows and, where the
// weights are many (from about 25 million a pair, 35 million a single product), at any count (choose_narrow8 has the rule).
// Us, tiled -> now, at 1 / 32 / 128 rows: pairs 512 x 1024 7.6 / 7.7 / 8.0 -> 3.6 / 4.2 / 4.8, 1024 x 2816 10.8 / 11.3 / 12.3 -> 4.1 / 5.8 / 7.1,
// 1536 x 4096 11.8 / 16.1 / 18.1 -> 5.2 / 7.2 / 10.5, 2048 x 5632 12.8 / 14.9 -> 10.2 / 10.0; single ones 1024 x 512 8.8 / 9.2 / 11.5 -> 2.4 / 3.0 / 3.1,
// 5632 x 2048 13.0 / 14.7 / 20.7 -> 6.1 / 8.1 / 13.2.  Whole FFN block: 1 x 512 x 1024 22.1 -> 12.0, 122 x 768 x 2816 29.3 -> 20.2, 8 x 1536 x 4096 34.6 -> 18.2,
// 16 x 2048 x 5632 33.8 -> 27.8.  The error against 64 bits is the tiled form's (1.3e-5 in norm at k 2816 to 11008).
// A non-temporal hint on weights that only one row of tiles reads was slower (1024 x 512, 1 row: 2.9 against 2.4).
#pragma once

#include <hip/hip_runtime.h>

namespace pto_hip {
namespace gemm8 {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float nf32x4;
typedef __attribute__((__vector_size__(8 * sizeof(int)))) int ni32x8;
typedef __attribute__((__vector_size__(4 * sizeof(int)))) int ni32x4;

// Tile of 16 MT rows x 16 CT channels (of both matrices of a pair); the workgroup's KW wavefronts take its steps of 128 codes
// in turn, NS of them in registers at once, and sum through LDS in wavefront order.  n % 4 == 0, k % 128 == 0.
template <bool DUAL, int CT, int MT, int KW, int NS, typename OutT>
__global__ __launch_bounds__(KW * 64) void narrow_gemm8_kernel(Params p, int tiles_n) {
  constexpr int MATS = DUAL ? 2 : 1, kStepK = 128;
  __shared__ __attribute__((aligned(16))) nf32x4 red[KW][MATS][CT][MT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int tn = blockIdx.x % tiles_n, tm = blockIdx.x / tiles_n;
  const int m0 = tm * 16 * MT, n0 = tn * 16 * CT;
  const int mine = (p.k / kStepK - wave + KW - 1) / KW;  // steps of this wavefront

  // a lane holds 32 codes of row (or channel) c, k = 32 kg .. of a step, of both operands alike
  const uint8_t* xp[MT];
  const uint8_t* wp[MATS][CT];
#pragma unroll
  for (int h = 0; h < MT; ++h) xp[h] = p.a + (size_t)min(m0 + 16 * h + c, p.m - 1) * p.lda + wave * kStepK + kg * 32;
#pragma unroll
  for (int t = 0; t < MATS; ++t)
#pragma unroll
    for (int i = 0; i < CT; ++i) wp[t][i] = (t ? p.b1 : p.b0) + (size_t)min(n0 + 16 * i + c, p.n - 1) * p.ldb + wave * kStepK + kg * 32;

  struct Held {
    ni32x4 w[MATS][CT][2], x[MT][2];
  };
  nf32x4 acc[MATS][CT][MT];
#pragma unroll
  for (int t = 0; t < MATS; ++t)
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
      for (int h = 0; h < MT; ++h) acc[t][i][h] = nf32x4{0.f, 0.f, 0.f, 0.f};
  // Past its last step a wavefront asks for its first again, one line a row (the requests in flight stay known at compile time).
  auto load = [&](Held& s, int round) {
    const size_t at = round < mine ? (size_t)round * KW * kStepK : 0;
#pragma unroll
    for (int t = 0; t < MATS; ++t)
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) s.w[t][i][q] = *reinterpret_cast<const ni32x4*>(wp[t][i] + at + q * 16);
#pragma unroll
    for (int h = 0; h < MT; ++h)
#pragma unroll
      for (int q = 0; q < 2; ++q) s.x[h][q] = *reinterpret_cast<const ni32x4*>(xp[h] + at + q * 16);
  };
  auto whole = [](const ni32x4 (&v)[2]) { return __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7); };
  auto compute = [&](const Held& s) {
#pragma unroll
    for (int h = 0; h < MT; ++h)
#pragma unroll
      for (int t = 0; t < MATS; ++t)
#pragma unroll
        for (int i = 0; i < CT; ++i)  // weights first: a lane then holds four consecutive channels of a row
          acc[t][i][h] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(whole(s.w[t][i]), whole(s.x[h]), acc[t][i][h], 0, 0, 0, 0, 0, 0);
  };
  Held st[NS];
  if (mine > 0) {
#pragma unroll
    for (int i = 0; i < NS - 1; ++i) load(st[i], i);
    int r = 0;
    for (; r + NS <= mine; r += NS) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        load(st[(i + NS - 1) % NS], r + i + NS - 1);
        compute(st[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < NS - 1; ++i)
      if (r + i < mine) compute(st[i]);
  }
#pragma unroll
  for (int t = 0; t < MATS; ++t)
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
      for (int h = 0; h < MT; ++h) red[wave][t][i][h][lane] = acc[t][i][h];
  __syncthreads();
  for (int u = tid; u < CT * MT * 64; u += KW * 64) {
    const int l = u & 63, h = (u >> 6) % MT, i = (u >> 6) / MT;
    const int row = m0 + 16 * h + (l & 15), col = n0 + 16 * i + 4 * (l >> 4);
    if (row >= p.m || col >= p.n) continue;
    nf32x4 sum[MATS];
#pragma unroll
    for (int t = 0; t < MATS; ++t) {
      sum[t] = red[0][t][i][h][l];
#pragma unroll
      for (int w = 1; w < KW; ++w) sum[t] += red[w][t][i][h][l];
    }
    const float r = p.sa[row];
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = sum[0][e] * r * p.sb0[col + e];
      if constexpr (DUAL) y[e] = silu(y[e]) * (sum[MATS - 1][e] * r * p.sb1[col + e]);
    }
    store4<OutT>(reinterpret_cast<OutT*>(p.c) + (int64_t)row * p.ldc + col, y);
  }
}

template <bool DUAL, int CT, int MT, int KW, int NS, typename OutT>
int launch_narrow8_tile(const Params& p, hipStream_t st) {
  const int tiles_n = (p.n + 16 * CT - 1) / (16 * CT), tiles_m = (p.m + 16 * MT - 1) / (16 * MT);
  hipLaunchKernelGGL((narrow_gemm8_kernel<DUAL, CT, MT, KW, NS, OutT>), dim3((unsigned)(tiles_n * tiles_m)), dim3(KW * 64), 0, st, p, tiles_n);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}
// tile: 1 to 3, as choose_narrow8 (launch_choice.h) numbers them.
template <bool DUAL, typename OutT>
int launch_narrow8(const Params& p, int tile, hipStream_t st) {
  if (tile == 1) return launch_narrow8_tile<DUAL, 1, 1, 4, 4, OutT>(p, st);
  if (tile == 2) return launch_narrow8_tile<DUAL, 2, 2, 4, 3, OutT>(p, st);
  return launch_narrow8_tile<DUAL, 2, 4, 8, DUAL ? 2 : 3, OutT>(p, st);
}

}  // namespace gemm8
}  // namespace pto_hip

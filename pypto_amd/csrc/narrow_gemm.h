// Products of a small call in one launch each: y[M, N] = x[M, K] @ W[K, N] (+ residual), or SiLU(x @ Wg) * (x @ Wu), W 16-bit values.
//
// Such a product is bound by its chain, not by bytes or MFMAs: the launch, one memory round trip per stage of the k loop, the
// stores, and with k split over workgroups a second launch that sums the slabs.  The tiled GEMM (gemm.h) stages 64 rows x 256
// columns through LDS: 128 rows of a 512 x 1024 pair are 16 workgroups that walk 16 stages one behind the other.
// Here a tile is 16 to 64 rows x 32 or 64 channels, so that a small product has a workgroup for every CU; the workgroup's
// wavefronts split k among themselves (no slabs, no second launch), and a wavefront with few steps requests all of
// them at once, one round trip.  Operands go straight to registers: a lane reads 8 or 4 bytes of 8 k rows (32- to 128-byte
// row pieces per 16 lanes) and transposes them with v_perm_b32 into MFMA operands, as the skinny projections do.  Every tile reads
// its operands for itself, which is why it stops paying at a few hundred rows (choose_narrow has the rule).
// Us, before (with the slabs' finish) -> now: 128 rows fp16 gate/up 512 x 1024 8.2 -> 4.3, 1024 x 512 8.7 -> 4.4, gate/up 1024 x 2048 15.5 ->
// 9.7, 2048 x 1024 10.8 -> 7.1, 1024 x 1024 9.5 -> 4.6; 512 rows gate/up 1024 x 2048 17.8 -> 13.5, 2048 x 2048 20.2 -> 15.1;
// ragged 1000 x 2504 pair at 96 rows 20.0 -> 10.4.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm.h"

namespace pto_hip {
namespace gemm {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef uint32_t u32x2 __attribute__((__vector_size__(2 * sizeof(uint32_t))));

constexpr int kNarrowStep = 32;  // k rows per step

template <bool BF16>
__device__ __forceinline__ f32x4 narrow_mfma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

template <int CH, int MATS, int MT>
struct NarrowStage {
  uint32_t w[MATS][8][CH / 2];  // CH channels of the k rows kg*8 .. kg*8+7
  u32x4 xa[MT];                 // activations of rows c + 16 h, k = kg*8 .. +8
};

// Tile of 16 MT rows x 16 CH channels (of both matrices of a pair); the workgroup's KW wavefronts take the tile's
// 32-row steps of k in turn and their accumulators are summed through LDS in wavefront order.  NS: steps a wavefront has
// in registers at once.  Eight wavefronts unless their sums outgrow the LDS (16 x 32 tile of a 1024-row k on 4 / 8 / 16: 4.6 / 4.4 / 4.6 us,
// 2048-row 7.0 / 7.1 / 6.8).
template <bool BF16, bool DUAL, int CH, int MT, int KW, int NS, typename OutT>
__global__ __launch_bounds__(KW * 64) void narrow_gemm_kernel(GemmParams p) {
  constexpr int MATS = DUAL ? 2 : 1;
  constexpr int kTile = 16 * CH, kRows = 16 * MT;
  typedef NarrowStage<CH, MATS, MT> Stage;
  __shared__ __attribute__((aligned(16))) float red[KW][MATS][kRows][kTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int tn = blockIdx.x % p.tiles_n, tm = blockIdx.x / p.tiles_n;
  const int m0 = tm * kRows, n0 = tn * kTile;
  const int steps = (p.k + kNarrowStep - 1) / kNarrowStep;

  size_t x_off[MT];
#pragma unroll
  for (int h = 0; h < MT; ++h) x_off[h] = (size_t)min(m0 + c + 16 * h, p.m - 1) * p.k + kg * 8;
  const size_t w_off = (size_t)(kg * 8) * p.n + min(n0 + c * CH, p.n - CH);

  f32x4 acc[MATS][CH][MT];
#pragma unroll
  for (int t = 0; t < MATS; ++t)
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int h = 0; h < MT; ++h) acc[t][i][h] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Loads are unconditional, so that the requests in flight are known at compile time: past its last step a wavefront asks
  // for one address over and over.  A last step that would reach past row k ends at row k; the rows it repeats are cleared in
  // both operands.
  const int mine = (steps - wave + KW - 1) / KW;  // steps of this wavefront
  auto load = [&](Stage& s, int round, auto all_real) {
    constexpr bool REAL = decltype(all_real)::value;
    const int mask = REAL ? -1 : (round - mine) >> 31;
    const int row0 = min((round * KW + wave) * kNarrowStep, p.k - kNarrowStep) & mask;
    const size_t lane_w = REAL ? w_off : w_off & (size_t)(int64_t)mask;
    const size_t pitch = REAL ? (size_t)p.n : (size_t)(uint32_t)(p.n & mask);
#pragma unroll
    for (int t = 0; t < MATS; ++t) {
      const uint16_t* w = (t ? p.b1 : p.b0) + (size_t)row0 * p.n + lane_w;
#pragma unroll
      for (int e = 0; e < 8; ++e) __builtin_memcpy(s.w[t][e], __builtin_assume_aligned(w + e * pitch, 2 * CH), 2 * CH);
    }
#pragma unroll
    for (int h = 0; h < MT; ++h)
      s.xa[h] = *reinterpret_cast<const u32x4*>(p.a + row0 + (REAL ? x_off[h] : x_off[h] & (size_t)(int64_t)mask));
  };
  auto compute = [&](Stage& s, int round) {
    const int step = round * KW + wave;
    if (step * kNarrowStep > p.k - kNarrowStep) {
      const uint32_t keep = p.k - kNarrowStep + kg * 8 >= step * kNarrowStep ? ~0u : 0u;
#pragma unroll
      for (int t = 0; t < MATS; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int j = 0; j < CH / 2; ++j) s.w[t][e][j] &= keep;
#pragma unroll
      for (int h = 0; h < MT; ++h) s.xa[h] &= u32x4{keep, keep, keep, keep};
    }
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int t = 0; t < MATS; ++t) {
        u32x4 b;
        const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = __builtin_amdgcn_perm(s.w[t][2 * q + 1][i >> 1], s.w[t][2 * q][i >> 1], sel);
#pragma unroll
        for (int h = 0; h < MT; ++h) acc[t][i][h] = narrow_mfma<BF16>(s.xa[h], b, acc[t][i][h]);
      }
  };
  // Up to NS steps: all of them requested at once, one round trip.
  Stage st[NS];
  auto at_once = [&](auto count) {
    constexpr int C = decltype(count)::value;
#pragma unroll
    for (int i = 0; i < C; ++i) load(st[i], i, std::true_type{});
#pragma unroll
    for (int i = 0; i < C; ++i) compute(st[i], i);
  };
  if (mine > NS) {
#pragma unroll
    for (int i = 0; i < NS - 1; ++i) load(st[i], i, std::true_type{});
    int r = 0;
    for (; r + NS <= mine; r += NS) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        load(st[(i + NS - 1) % NS], r + i + NS - 1, std::false_type{});
        compute(st[i], r + i);
      }
    }
#pragma unroll
    for (int i = 0; i < NS - 1; ++i)
      if (r + i < mine) compute(st[i], r + i);
  } else if (NS >= 4 && mine == 4) at_once(std::integral_constant<int, NS >= 4 ? 4 : 1>{});
  else if (NS >= 3 && mine == 3) at_once(std::integral_constant<int, NS >= 3 ? 3 : 1>{});
  else if (mine == 2) at_once(std::integral_constant<int, 2>{});
  else if (mine == 1) at_once(std::integral_constant<int, 1>{});

  // acc[t][i][h][r] is row 16 h + 4 kg + r, channel c CH + i
#pragma unroll
  for (int t = 0; t < MATS; ++t)
#pragma unroll
    for (int h = 0; h < MT; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = acc[t][i][h][r];
        __builtin_memcpy(__builtin_assume_aligned(&red[wave][t][16 * h + 4 * kg + r][c * CH], 4 * CH), v, 4 * CH);
      }
  __syncthreads();
  constexpr int kQuads = kTile / 4;
  for (int u = tid; u < kRows * kQuads; u += KW * 64) {
    const int row = u / kQuads, q = u % kQuads;
    const int m = m0 + row, n = n0 + 4 * q;
    if (m >= p.m || n >= p.n) continue;
    f32x4 sum[MATS];
#pragma unroll
    for (int t = 0; t < MATS; ++t) {
      sum[t] = *reinterpret_cast<const f32x4*>(&red[0][t][row][4 * q]);
#pragma unroll
      for (int w = 1; w < KW; ++w) sum[t] += *reinterpret_cast<const f32x4*>(&red[w][t][row][4 * q]);
    }
    OutT* out = reinterpret_cast<OutT*>(p.c) + (int64_t)m * p.ldc + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float y = sum[0][j];
      if constexpr (DUAL) y = silu(y) * sum[MATS - 1][j];
      else if (p.residual) y += load_residual(p.residual, p.res_dtype, (int64_t)m * p.n + n + j);
      store_out<OutT>(out + j, y);
    }
  }
}

template <bool BF16, bool DUAL, int CH, int MT, int KW, int NS, typename OutT>
int launch_narrow_tile(GemmParams p, hipStream_t st) {
  p.tiles_n = (p.n + 16 * CH - 1) / (16 * CH);
  p.tiles_m = (p.m + 16 * MT - 1) / (16 * MT);
  hipLaunchKernelGGL((narrow_gemm_kernel<BF16, DUAL, CH, MT, KW, NS, OutT>), dim3((unsigned)(p.tiles_n * p.tiles_m)), dim3(KW * 64), 0, st, p);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

// tile: 1 to 4, as choose_narrow (launch_choice.h) numbers them.
template <bool BF16, bool DUAL, typename OutT>
int launch_narrow(const GemmParams& p, int tile, hipStream_t st) {
  switch (tile) {
    case 1: return launch_narrow_tile<BF16, DUAL, 2, 1, 8, 4, OutT>(p, st);
    case 2: return launch_narrow_tile<BF16, DUAL, 2, 2, 8, 4, OutT>(p, st);
    case 3: return launch_narrow_tile<BF16, DUAL, 4, 2, 8, DUAL ? 3 : 4, OutT>(p, st);
    default: return launch_narrow_tile<BF16, DUAL, 4, 4, DUAL ? 4 : 8, 3, OutT>(p, st);
  }
}

}  // namespace gemm
}  // namespace pto_hip

// Projections of some tens of rows that are bound by reading their weights: y[M, N] = x[M, K] @ W[K, N], W int8 codes or 16-bit
// values, M up to 96, left as fp32 slabs of k splits for the kernel that follows.
//
// The tiled GEMM multiplies such a batch on 64- or 128-row tiles 256 columns wide and takes its codes through registers and LDS;
// here a weight goes from memory to the registers of the one wavefront that multiplies it, as in the skinny projections
// (skinny.h), whose loop this is with 3, 4 or 6 groups of 16 rows.  What bounds it: a CU's L1 takes about four clocks per 128-byte
// line, and beside the weights it has to take in every activation once per 128 channels.  Hence the blocked layout - a
// wavefront's 1 KB of activations is 8 whole lines, in rows it is 16 halves (96 rows of int8 4096 x 14336 pairs 40 us, in rows 50, without
// any activations 30.5) - and one 128-channel slab a workgroup: two slabs sharing their activations through L1 38.5 us but twice the
// partial sums.  More than two stages in flight change nothing (2 / 3 / 4 / 5 stages 40.1 / 40.9 / 40.3 / 41.5), but three at 96 rows of 16-bit
// weights (54.0 -> 49.9).  Activations staged in rows through LDS for two slabs at once: 40.7 us, 16-bit 45.9 for 49.9, but 13.1 for 10.9 in a
// 4096 x 4096 product; eight row groups (128 rows) 45 us, level with the tiled GEMM.
#pragma once

#include "skinny.h"

namespace pto_hip {
namespace stream {

using namespace skinny;

struct StreamParams {
  const uint16_t* x;  // [M, K] 16-bit activations, or [K/8][x_rows][8]
  const void* w[2];   // [K, N] each; the second is the up projection of a pair
  float* part;        // [mats][splits][M, N]
  int m, k, n, x_rows;
  int slabs, ks, splits, mats;  // 128-channel slabs of one matrix, 32-row steps of k
};

template <bool W8, int MT>
struct Held {
  typename std::conditional<W8, u32x2, u32x4>::type w[8];  // 8 channels of the k rows kg*8 .. kg*8+7
  u32x4 xa[MT];                                            // activations of rows c + 16 h, k = kg*8 .. +8
};

// Workgroup = (slab of 128 channels, k split); its four wavefronts, one per SIMD, take the split's steps in turn and sum
// their accumulators (MT x 8 tiles of 16 x 16, up to 192 registers) through LDS.  NS register stages.
template <bool BF16, bool W8, int MT, int NS>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 1))) void stream_rows_kernel(StreamParams p) {
  constexpr int kCols = 8, kSlab = 16 * kCols, kWBytes = W8 ? 1 : 2;
  typedef typename std::conditional<W8, u32x2, u32x4>::type wvec_t;
  extern __shared__ __attribute__((aligned(16))) float red[];  // [2][kWaves][32][kSlab]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int split = blockIdx.x % p.splits, slab = blockIdx.x / p.splits;
  const int mat = slab >= p.slabs ? 1 : 0;
  const int nb = (slab - mat * p.slabs) * kSlab;  // the slab's first channel
  const int s0 = (int)((int64_t)p.ks * split / p.splits), s1 = (int)((int64_t)p.ks * (split + 1) / p.splits);
  const int rounds = (s1 - s0 + kWaves - 1) / kWaves;

  const int x_step = p.x_rows ? p.x_rows : 1;  // elements per unit of k
  uint32_t x_off[MT];                          // bytes
#pragma unroll
  for (int h = 0; h < MT; ++h) {
    const uint32_t row = (uint32_t)min(c + 16 * h, p.m - 1);
    x_off[h] = (p.x_rows ? ((uint32_t)(kg * p.x_rows) + row) * 8u : row * (uint32_t)p.k + (uint32_t)(kg * 8)) * 2u;
  }
  const size_t w_off = ((size_t)(kg * 8) * p.n + min(nb + c * kCols, p.n - kCols)) * kWBytes;
  const char* const wmat = reinterpret_cast<const char*>(p.w[mat]);
  const char* const x = reinterpret_cast<const char*>(p.x);

  f32x4 acc[kCols][MT];
#pragma unroll
  for (int i = 0; i < kCols; ++i)
#pragma unroll
    for (int h = 0; h < MT; ++h) acc[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Loads never depend on a condition, so that the requests in flight are known at compile time: past its last step a
  // wavefront asks for one address over and over.  A last step that would reach past row k ends at row k; the rows it then repeats
  // are cleared in the activations, and in 16-bit weights too: an infinity there must not become a NaN.
  auto load = [&](Held<W8, MT>& s, int round) {
    const int step = s0 + round * kWaves + wave;
    const bool real = step < s1;
    const int row0 = real ? min(step * kStep, p.k - kStep) : 0;
    const char* const wbase = real ? wmat + (size_t)row0 * p.n * kWBytes : x;
    const size_t pitch = real ? (size_t)p.n * kWBytes : 0;
    const size_t off = real ? w_off : 0;
    const char* const xbase = x + (size_t)row0 * x_step * 2;
#pragma unroll
    for (int e = 0; e < 8; ++e) s.w[e] = __builtin_nontemporal_load(reinterpret_cast<const wvec_t*>(wbase + e * pitch + off));
#pragma unroll
    for (int h = 0; h < MT; ++h) s.xa[h] = *reinterpret_cast<const u32x4*>(xbase + x_off[h]);
  };
  auto compute = [&](const Held<W8, MT>& s, int round) {
    const int step = s0 + round * kWaves + wave;
    if (step >= s1) return;  // uniform
    const bool k_ok = min(step * kStep, p.k - kStep) + kg * 8 >= step * kStep;
    multiply<BF16, W8, kCols, MT>(s.w, s.xa, k_ok, acc);
  };
  Held<W8, MT> st[NS];
#pragma unroll
  for (int i = 0; i < NS - 1; ++i) load(st[i], i);
  for (int r = 0; r < rounds; r += NS) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      load(st[(i + NS - 1) % NS], r + i + NS - 1);
      compute(st[i], r + i);
    }
  }

  // 32 rows at a time through LDS, two areas in turn; float4s of a row in the order (v, c) as in store_run
  constexpr int kQuads = kSlab / 4;
  const int q = tid % kQuads, n = nb + (q & 15) * kCols + (q >> 4) * 4;
  float* const out = p.part + ((size_t)mat * p.splits + split) * p.m * p.n + n;
#pragma unroll
  for (int h0 = 0; h0 < MT; h0 += 2) {
    constexpr int kRows = 32;
    float4* const buf = reinterpret_cast<float4*>(red) + ((h0 >> 1) & 1) * (kWaves * kRows * kQuads);
    float4* const mine = buf + wave * (kRows * kQuads) + c;
#pragma unroll
    for (int h = h0; h < h0 + 2 && h < MT; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int v = 0; v < kCols / 4; ++v)
          mine[((h - h0) * 16 + 4 * kg + r) * kQuads + v * 16] =
              float4{acc[4 * v][h][r], acc[4 * v + 1][h][r], acc[4 * v + 2][h][r], acc[4 * v + 3][h][r]};
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (n < p.n) {
      const int rows = min(p.m - 16 * h0, min(kRows, 16 * (MT - h0)));
      for (int row = tid / kQuads; row < rows; row += kWaves * 64 / kQuads) {
        const float4* src = buf + row * kQuads + q;
        float4 a = src[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
          const float4 v = src[w * (kRows * kQuads)];
          a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w;
        }
        *reinterpret_cast<float4*>(out + (size_t)(16 * h0 + row) * p.n) = a;
      }
    }
  }
}

template <bool BF16, bool W8, int MT, int NS>
int launch_rows(const StreamParams& p, hipStream_t st) {
  constexpr int kLds = 2 * kWaves * 32 * 128 * (int)sizeof(float);
  auto kern = stream_rows_kernel<BF16, W8, MT, NS>;
  static std::atomic<bool> attr_set{false};  // per instantiation; callers hold the dispatch lock
  if (!attr_set.load(std::memory_order_acquire)) {
    PTO_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    attr_set.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.slabs * p.mats * p.splits)), dim3(kWaves * 64), kLds, st, p);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}
template <bool BF16>
int launch_w8(const StreamParams& p, hipStream_t st) {
  if (p.m <= 48) return launch_rows<BF16, true, 3, 2>(p, st);
  if (p.m <= 64) return launch_rows<BF16, true, 4, 2>(p, st);
  return launch_rows<BF16, true, 6, 2>(p, st);
}
template <bool BF16>
int launch_w16(const StreamParams& p, hipStream_t st) {
  if (p.m <= 48) return launch_rows<BF16, false, 3, 2>(p, st);
  if (p.m <= 64) return launch_rows<BF16, false, 4, 2>(p, st);
  return launch_rows<BF16, false, 6, 3>(p, st);
}

}  // namespace stream
}  // namespace pto_hip

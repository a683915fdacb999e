// W8A16 decode projections: y[M<=32, N] = (x[M, K] @ Wq[K, N]) * scale[N], Wq int8 stored [in, out].
//
// The reference has no quantised-weight path; this follows its projection kernels' contract
// (x @ W with W [in, out] row-major, fp32 accumulation, examples/models/qwen3_jit/kernels/
// projection.py:145-177) with int8 weights and one fp32 scale per output channel.  Decode
// batches are small (M <= 32), so the work is reading the weights once: HBM-bound.
//
//   * the (128- or 256-channel slab, 32-row step) units of a launch are shared out evenly over workgroups of
//     four wavefronts, at most one per CU, and whole numbers of them to a slab where that keeps most CUs
//     busy (skinny_workgroups); the wavefronts take a share's steps in turn.  Per step a lane reads 8 or 16 bytes of 8
//     k-rows - whole row segments per 16 lanes - keeps the next step's loads in flight,
//     widens the int8 codes to fp32 and packs them, transposed, straight into MFMA B operands
//     (the high halves of the fp32 values are exact bf16), then issues its v_mfma_f32_16x16x32;
//   * at the end of a slab's share the four accumulators are summed through LDS in a fixed order and
//     written as one fp32 partial slab;
//   * the partial slabs are summed in order, scaled per channel and finished by a small
//     second kernel: residual add / SwiGLU / cast, or residual add + RMSNorm of the whole row.
//     The RoPE kernel reads the q/k/v partials directly.
// Launch and finish, cold weights, 16 rows: 16 MB of 16-bit weights 11.3 us, 356 MB 63 us (5.7 TB/s); int8 117 MB 26 us.
// In the decoder layer (trace, equal k ranges on the CUs and 32 rows always before -> now): one sequence, int8
// q/k/v 11.0 -> 8.5 us, o 10.1 -> 8.0, gate/up 25.7 -> 22.9, down 13.6 -> 12.4; sixteen sequences, 16-bit weights of a 5120-wide
// model: q/k/v 16.5 -> 14.6, o 13.2 -> 12.2, gate/up 76.0 -> 59.8, down 34.2 -> 32.4; steps 84 -> 75 and 188 -> 169 us,
// 32 sequences int8 (two row groups) 163.6 -> 161.0.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.h"
#include "launch_choice.h"
#include "slab_sum.h"

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;

constexpr int kStep = 32;                // k rows per step
constexpr int kMaxM = pto_hip::kW8MaxM;
constexpr int kWaves = 4;                // wavefronts per workgroup of the partial kernel

struct GemvParams {
  const uint16_t* x;    // [M, K] 16-bit activations
  const void* wq[2];    // [K, N] each (int8 codes or 16-bit weights); the second is the up projection of a pair
  float* part[2];       // [partial slabs, M, N] each
  int m, k, n, x_blocked;  // x_blocked: activations stored [K/8][32][8] (see w8a16_partials) instead of row-major
  int slabs, ks;        // output slabs of one matrix, 32-row steps of one slab
  int per_wg, extra;    // units / workgroups and its remainder (see SlabMap)
  int mapped;           // 0: a workgroup per slab
};

template <bool BF16>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

// Two small integers held as fp32 -> packed pair of 16-bit floats, exact.
template <bool BF16>
__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  if constexpr (BF16) {
    // |value| <= 128 has at most 8 significant bits: the upper half of the fp32 pattern is the bf16.
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo),
                                 0x07060302u);
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
  }
}

typedef uint32_t u32x2 __attribute__((__vector_size__(2 * sizeof(uint32_t))));

// One register stage of a lane: kCols channels of the k rows kg*8 .. kg*8+7, and the activations.
// W8: int8 weight codes, 8 bytes (kCols 8) or 16 bytes (kCols 16) per row and lane; otherwise
// 16-bit weights of the activation type (16 bytes = 8 channels).
template <bool W8, int kCols, int MT>
struct Stage {
  typename std::conditional<(W8 && kCols == 8), u32x2, u32x4>::type w[8];
  u32x4 xa[MT];  // activations of rows c (and c+16), k = kg*8 .. +8
};

// Workgroup w of G takes the units (slab, 32-row step) [w U / G, (w + 1) U / G) of the list that walks the
// slabs one after the other (SlabMap): every workgroup streams the same number of bytes.  A launch lasts as
// long as the CU with the most bytes: cut into equal k ranges instead, 272 workgroups of a 356 MB pair of 16-bit
// matrices on 256 CUs read at 4.5 TB/s and 544 at 5.3, where 256 even shares reach 6.5 (load-only twins of
// this kernel).  The four wavefronts take a run's steps in turn; when
// a run ends (the slab's last step or the workgroup's) their accumulators are summed through LDS, one after
// the other, and written as the next partial slab of those channels; the next run's first rows
// are in flight meanwhile.  MT: 16-row groups of activations (M <= 16 needs one: half the MFMAs,
// activations and partial sums).  Rows past M are computed on row M - 1 and not written.
template <bool BF16, bool W8, int kCols, int MT, bool NT>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 2))) void w8a16_partial_kernel(GemvParams p) {
  static_assert(kCols == 8 || (W8 && kCols == 16), "16 channels per lane only with int8 codes");
  constexpr int kSlab = 16 * kCols;  // output channels of a slab: 16 lanes of kCols channels
  constexpr int kRows = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) float red[];  // [kWaves][kRows][kSlab]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: row addresses stay scalar
  const int c = lane & 15, kg = lane >> 4;

  // this workgroup's units, and a cursor over them in rounds of kWaves steps of one slab
  const int wg = blockIdx.x, wgs = gridDim.x;
  const int u_begin = wg * p.per_wg + wg * p.extra / wgs, u_end = (wg + 1) * p.per_wg + (wg + 1) * p.extra / wgs;
  struct Cursor {
    int slab, step, end;  // the round's first step and the end of its run
  };
  auto run_end = [&](int slab) { return min(p.ks, u_end - slab * p.ks); };
  auto last_of_run = [&](const Cursor& cur) { return cur.step + kWaves >= cur.end; };
  auto last = [&](const Cursor& cur) { return last_of_run(cur) && cur.slab * p.ks + cur.end >= u_end; };
  auto advance = [&](Cursor& cur) {
    if (!last_of_run(cur)) {
      cur.step += kWaves;
    } else {
      cur.slab += 1;
      cur.step = 0;
      cur.end = run_end(cur.slab);
    }
  };

  // Row-major x: lane (c, kg) reads 16 bytes of rows c and c+16 at k = kstep + 8*kg.  Blocked x
  // keeps the 32 rows of each 8-k group together, so the same reads of a wavefront cover
  // consecutive bytes instead of half cache lines.
  const int x_step = p.x_blocked ? kMaxM : 1;  // elements per unit of k
  const uint16_t* xp[MT];
#pragma unroll
  for (int h = 0; h < MT; ++h) {
    const int row = min(c + 16 * h, p.m - 1);
    xp[h] = p.x_blocked ? p.x + (size_t)(kg * kMaxM + row) * 8 : p.x + (size_t)row * p.k + kg * 8;
  }

  f32x4 acc[kCols][MT];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < kCols; ++i)
#pragma unroll
      for (int h = 0; h < MT; ++h) acc[i][h] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();

  // Loads never depend on a condition, so the number of requests in flight is known at compile
  // time: a wavefront without a step of its own in a round reads the run's last one again, and a last step
  // that would reach past row k is moved back to end at row k - the rows it then repeats are
  // multiplied by zeroed activations.  A row address is a wavefront-uniform row base plus a
  // per-lane offset.
  constexpr int kWBytes = W8 ? 1 : 2;  // bytes per weight
  typedef typename std::conditional<(W8 && kCols == 8), u32x2, u32x4>::type wvec_t;
  auto load = [&](Stage<W8, kCols, MT>& s, const Cursor& cur) {
    const int row0 = min(min(cur.step + wave, cur.end - 1) * kStep, p.k - kStep);
    const int mat = cur.slab >= p.slabs ? 1 : 0;
    const int n0 = min((cur.slab - mat * p.slabs) * kSlab + c * kCols, p.n - kCols);
    const size_t lane_off = ((size_t)n0 + (size_t)(kg * 8) * p.n) * kWBytes;
    const char* wbase = reinterpret_cast<const char*>(p.wq[mat]) + (size_t)row0 * p.n * kWBytes;
#pragma unroll
    for (int h = 0; h < MT; ++h) s.xa[h] = *reinterpret_cast<const u32x4*>(xp[h] + (size_t)row0 * x_step);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const char* row = wbase + (size_t)e * p.n * kWBytes;  // uniform
      if constexpr (NT) s.w[e] = __builtin_nontemporal_load(reinterpret_cast<const wvec_t*>(row + lane_off));
      else s.w[e] = *reinterpret_cast<const wvec_t*>(row + lane_off);
    }
  };
  auto compute = [&](const Stage<W8, kCols, MT>& s, const Cursor& cur) {
    const int step = cur.step + wave;
    if (step >= cur.end) return;  // uniform: no step for this wavefront in this round
    const bool k_ok = min(step * kStep, p.k - kStep) + kg * 8 >= step * kStep;
    u32x4 a[MT];
#pragma unroll
    for (int h = 0; h < MT; ++h) a[h] = k_ok ? s.xa[h] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
      // channel n0 + i: its 8 k-values, as packed pairs (k, k+1)
      u32x4 b;
      if constexpr (W8) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t w0 = s.w[2 * q][i >> 2];
          const uint32_t w1 = s.w[2 * q + 1][i >> 2];
          const float f0 = (float)(int8_t)(w0 >> ((i & 3) * 8));
          const float f1 = (float)(int8_t)(w1 >> ((i & 3) * 8));
          b[q] = pack_pair<BF16>(f0, f1);
        }
      } else {
        // 16-bit weights: element i of rows 2q and 2q+1 (an 8x8 transpose in registers)
        const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = __builtin_amdgcn_perm(s.w[2 * q + 1][i >> 1], s.w[2 * q][i >> 1], sel);
      }
#pragma unroll
      for (int h = 0; h < MT; ++h) acc[i][h] = mfma16<BF16>(a[h], b, acc[i][h]);
      __builtin_amdgcn_sched_barrier(0);  // keep the conversions next to their MFMAs
    }
  };

  // End of a run: the wavefronts' accumulators through LDS into one partial slab.  acc[i][h][r] is row
  // h*16 + 4*kg + r, channel c*kCols + i; the float4s of a row are kept in the order (v, c) - channels c*kCols + 4v .. -
  // so that neither the writes nor the reads of 16 lanes collide in a bank.
  constexpr int kQuads = kSlab / 4;
  auto finish_run = [&](const Cursor& cur) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the last run's sums have been read
    float4* mine = reinterpret_cast<float4*>(red) + wave * (kRows * kQuads) + c;
#pragma unroll
    for (int h = 0; h < MT; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int v = 0; v < kCols / 4; ++v)
          mine[(h * 16 + 4 * kg + r) * kQuads + v * 16] =
              float4{acc[4 * v][h][r], acc[4 * v + 1][h][r], acc[4 * v + 2][h][r], acc[4 * v + 3][h][r]};
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int mat = cur.slab >= p.slabs ? 1 : 0;
    // partial slab number: how many workgroups before this one hold steps of the slab (the one
    // that holds its first unit has number 0)
    const int first = cur.slab * p.ks;
    const int owner = p.mapped ? (int)(((unsigned)(first + 1) * (unsigned)wgs - 1) / (unsigned)(p.per_wg * wgs + p.extra)) : wg;
    const int q = tid % kQuads, n = (cur.slab - mat * p.slabs) * kSlab + (q & 15) * kCols + (q >> 4) * 4;
    float* out = p.part[mat] + (size_t)(wg - owner) * p.m * p.n + n;
    if (n < p.n) {
      for (int row = tid / kQuads; row < p.m; row += kWaves * 64 / kQuads) {
        const float4* src = reinterpret_cast<const float4*>(red) + row * kQuads + q;
        float4 a = src[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
          const float4 v = src[w * (kRows * kQuads)];
          a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w;
        }
        *reinterpret_cast<float4*>(out + (size_t)row * p.n) = a;
      }
    }
    clear();
  };

  Cursor use, ahead;
  use.slab = u_begin / p.ks;
  use.step = u_begin - use.slab * p.ks;
  use.end = run_end(use.slab);
  ahead = use;
  // Two register stages, one of them in flight while the other is multiplied (three and four measured slower: one
  // sequence's layer 75.2 -> 77.8 / 79.2 us).  The last round is a copy of its own that requests nothing:
  // behind a branch around the loads the compiler would wait for all of them in every round, and reading
  // the last rows again costs as much as a new round.
  Stage<W8, kCols, MT> st[2];
  load(st[0], ahead);
  auto round = [&](const Stage<W8, kCols, MT>& cur) {
    compute(cur, use);
    if (last_of_run(use)) finish_run(use);
  };
  for (;;) {
    if (last(use)) {
      round(st[0]);
      break;
    }
    advance(ahead);
    load(st[1], ahead);
    round(st[0]);
    advance(use);
    if (last(use)) {
      round(st[1]);
      break;
    }
    advance(ahead);
    load(st[0], ahead);
    round(st[1]);
    advance(use);
  }
}

struct FinishParams {
  const float* part0;   // [splits, 32 or M, N]: `stride` elements between splits
  const float* part1;   // second projection for SwiGLU, or null
  const float* scale0;  // [N]
  const float* scale1;
  const void* residual; // [M, N] in res_dtype, or null
  void* out;            // [M, N]
  int m, n, splits, res_dtype, out_dtype;
  int out_blocked;  // write out as [N/8][32][8] for the next projection
  int64_t stride;
  pto_hip::SlabMap map;
};

// Element index of (row m, channel n) in the blocked activation layout [N/8][32][8].
__device__ __forceinline__ size_t blocked_index(int m, int n) { return ((size_t)(n >> 3) * kMaxM + m) * 8 + (n & 7); }

__device__ __forceinline__ float4 load4_as_f32(const void* p, size_t i, int dt) {
  if (dt == PTO_HIP_FP32) return *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p) + i);
  const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint16_t*>(p) + i);
  if (dt == PTO_HIP_BF16)
    return float4{__builtin_bit_cast(float, v.x << 16), __builtin_bit_cast(float, v.x & 0xffff0000u),
                  __builtin_bit_cast(float, v.y << 16), __builtin_bit_cast(float, v.y & 0xffff0000u)};
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const h2 a = __builtin_bit_cast(h2, v.x), b = __builtin_bit_cast(h2, v.y);
  return float4{(float)a.x, (float)a.y, (float)b.x, (float)b.y};
}
__device__ __forceinline__ void store4_from_f32(void* p, size_t i, int dt, float4 v) {
  if (dt == PTO_HIP_FP32) {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(p) + i) = v;
  } else if (dt == PTO_HIP_BF16) {
    typedef __bf16 b4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<b4*>(reinterpret_cast<__bf16*>(p) + i) = b4{(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
  } else {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<h4*>(reinterpret_cast<_Float16*>(p) + i) =
        h4{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
  }
}

// Sums of the k splits of four channels of K matrices with `splits` slabs each, in split order, times the channel scales.
template <int K>
__device__ __forceinline__ void sum_splits(const float* const (&part)[K], const float* const (&scale)[K], int splits,
                                           size_t stride, int m, int n, int nn, f32x4 (&sum)[K]) {
  const float* src[K];
  f32x4 sc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    src[k] = part[k] + (size_t)m * nn + n;
    sum[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    sc[k] = scale[k] ? *reinterpret_cast<const f32x4*>(scale[k] + n) : f32x4{1.f, 1.f, 1.f, 1.f};  // none: unquantised weights
  }
  pto_hip::add_slabs(src, splits, stride, sum);
#pragma unroll
  for (int k = 0; k < K; ++k) sum[k] *= sc[k];
}
__device__ __forceinline__ float4 sum_splits(const float* part, const float* scale, int splits, size_t stride, int m,
                                             int n, int nn) {
  const float* parts[1] = {part};
  const float* scales[1] = {scale};
  f32x4 sum[1];
  sum_splits<1>(parts, scales, splits, stride, m, n, nn, sum);
  return float4{sum[0][0], sum[0][1], sum[0][2], sum[0][3]};
}

__device__ __forceinline__ float silu_mul(float g, float u) {
  return g * __frcp_rn(1.f + __expf(-g)) * u;  // SiLU(gate) * up, device form of 01_ffn.py:70-75
}

__global__ __launch_bounds__(256) void w8a16_finish_kernel(FinishParams p) {
  const int n = (blockIdx.x * 256 + threadIdx.x) * 4;
  const int m = blockIdx.y;
  if (n >= p.n) return;
  const size_t idx = (size_t)m * p.n + n;
  float4 r = {0.f, 0.f, 0.f, 0.f};  // requested with the slabs
  if (p.residual) r = load4_as_f32(p.residual, idx, p.res_dtype);
  const int splits0 = pto_hip::slab_count(p.map, p.splits, 0, n);
  float4 a;
  if (p.part1) {
    const int splits1 = pto_hip::slab_count(p.map, p.splits, 1, n);
    float4 u;
    if (splits0 == splits1) {
      const float* parts[2] = {p.part0, p.part1};
      const float* scales[2] = {p.scale0, p.scale1};
      f32x4 sum[2];
      sum_splits<2>(parts, scales, splits0, (size_t)p.stride, m, n, p.n, sum);
      a = float4{sum[0][0], sum[0][1], sum[0][2], sum[0][3]};
      u = float4{sum[1][0], sum[1][1], sum[1][2], sum[1][3]};
    } else {
      a = sum_splits(p.part0, p.scale0, splits0, (size_t)p.stride, m, n, p.n);
      u = sum_splits(p.part1, p.scale1, splits1, (size_t)p.stride, m, n, p.n);
    }
    a = float4{silu_mul(a.x, u.x), silu_mul(a.y, u.y), silu_mul(a.z, u.z), silu_mul(a.w, u.w)};
  } else {
    a = sum_splits(p.part0, p.scale0, splits0, (size_t)p.stride, m, n, p.n);
  }
  if (p.residual) {
    a.x += r.x; a.y += r.y; a.z += r.z; a.w += r.w;
  }
  store4_from_f32(p.out, p.out_blocked ? blocked_index(m, n) : idx, p.out_dtype, a);
}

// Finish of a projection followed by RMSNorm of the sum with the residual: one workgroup per
// row, the row (n <= 4 * kNormThreads * kNormVec channels) kept in registers between the two passes.
// Writes the fp32 sum (the next residual) and the normalised row.
constexpr int kNormVec = 2;
constexpr int kNormThreads = 1024;
struct FinishNormParams {
  const float* part;
  const float* scale;
  const void* residual;  // [M, N] in res_dtype
  float* sum_out;        // [M, N] fp32
  const float* gamma;    // [N]
  void* normed_out;      // [M, N] in out_dtype
  int n, splits, res_dtype, out_dtype;
  int out_blocked;
  float eps;
  int64_t stride;  // elements between splits
  pto_hip::SlabMap map;
};

__global__ __launch_bounds__(kNormThreads) void w8a16_finish_norm_kernel(FinishNormParams p) {
  const int m = blockIdx.x;
  float4 v[kNormVec];
  float4 g[kNormVec];  // requested with the row, so that the second pass waits for nothing
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < kNormVec; ++u) {
    const int n = (threadIdx.x + u * kNormThreads) * 4;
    if (n < p.n) {
      g[u] = *reinterpret_cast<const float4*>(p.gamma + n);
      const float4 r = load4_as_f32(p.residual, (size_t)m * p.n + n, p.res_dtype);
      float4 a = sum_splits(p.part, p.scale, pto_hip::slab_count(p.map, p.splits, 0, n), (size_t)p.stride, m, n, p.n);
      a.x += r.x; a.y += r.y; a.z += r.z; a.w += r.w;
      v[u] = a;
      *reinterpret_cast<float4*>(p.sum_out + (size_t)m * p.n + n) = a;
      ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  __shared__ float wsum[kNormThreads / 64];
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < kNormThreads / 64; ++w) tot += wsum[w];
  const float inv = rsqrtf(tot / (float)p.n + p.eps);
#pragma unroll
  for (int u = 0; u < kNormVec; ++u) {
    const int n = (threadIdx.x + u * kNormThreads) * 4;
    if (n < p.n) {
      const float4 y = {v[u].x * inv * g[u].x, v[u].y * inv * g[u].y, v[u].z * inv * g[u].z, v[u].w * inv * g[u].w};
      store4_from_f32(p.normed_out, p.out_blocked ? blocked_index(m, n) : (size_t)m * p.n + n, p.out_dtype, y);
    }
  }
}

template <typename P>
P* byte_offset(P* base, int64_t bytes) {
  return reinterpret_cast<P*>(reinterpret_cast<uintptr_t>(base) + (uintptr_t)bytes);
}

int check_common(const char* what, int64_t m, int64_t k, int64_t n, int x_dtype, int out_dtype) {
  using namespace pto_hip;
  PTO_CHECK_ARG(m >= 0 && m < (1 << 20), "%s: M = %lld rows out of range", what, (long long)m);
  PTO_CHECK_ARG(k >= kStep && k % 16 == 0, "%s: K = %lld must be a multiple of 16, at least %d", what,
                (long long)k, kStep);
  PTO_CHECK_ARG(n >= 8 && n % 8 == 0, "%s: N = %lld must be a positive multiple of 8", what, (long long)n);
  PTO_CHECK_ARG(k < (1 << 30) && n < (1 << 30), "%s: shape too large", what);
  PTO_CHECK_ARG(x_dtype == PTO_HIP_BF16 || x_dtype == PTO_HIP_FP16, "%s: x dtype %s not in {BF16, FP16}",
                what, dtype_name(x_dtype));
  PTO_CHECK_ARG(out_dtype == PTO_HIP_FP32 || out_dtype == PTO_HIP_BF16 || out_dtype == PTO_HIP_FP16,
                "%s: out dtype %s not in {FP32, BF16, FP16}", what, dtype_name(out_dtype));
  return PTO_HIP_OK;
}

template <bool BF16, bool W8, int kCols, int MT>
int launch_partial(const GemvParams& p, int wgs, bool nt, hipStream_t st) {
  const size_t smem = (size_t)kWaves * 16 * MT * 16 * kCols * sizeof(float);
  auto kern = nt ? w8a16_partial_kernel<BF16, W8, kCols, MT, true> : w8a16_partial_kernel<BF16, W8, kCols, MT, false>;
  static std::atomic<bool> attr_set[2];  // per instantiation; callers hold the dispatch lock
  if (!attr_set[nt].load(std::memory_order_acquire)) {
    PTO_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    attr_set[nt].store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(kWaves * 64), smem, st, p);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

}  // namespace

namespace pto_hip {

int w8a16_partials(const void* x, bool x_blocked, const void* wq0, const void* wq1, int64_t m, int64_t k, int64_t n,
                   int x_dtype, hipStream_t st, W8Partials* out, bool w16) {
  GemvParams p{};
  p.x = reinterpret_cast<const uint16_t*>(x);
  p.wq[0] = wq0;
  p.wq[1] = wq1;
  p.m = (int)m;
  p.k = (int)k;
  p.n = (int)n;
  p.x_blocked = x_blocked ? 1 : 0;
  const Context& cx = ctx();
  const int n_mats = wq1 ? 2 : 1;
  // int8 codes are read 16 per lane (256-channel slabs, 256-byte row pieces instead of 128) when rows and base
  // addresses allow 16-byte loads and the matrices are large.  Twice the channels in a slab are twice the partial
  // sums at the same number of workgroups, and 32 instead of 16 KB per wavefront through LDS at the end of a run.
  // Measured with their finish at 1 / 16 / 32 rows: 178 MB 36.0 / 38.8 / 44.6 us (8 per lane: 36.4 / 42.0 / 50.2), 117 MB
  // 24.1 / 26.0 / 29.6 (25.6 / 29.2 / 34.0), 89 MB 20.4 / 22.1 / 25.7 (21.9 / 24.9 / 28.6); but 67 MB 16.5 / 18.2 / 21.7
  // (15.6 / 17.7 / 20.7), 59 MB 15.8 / 17.5 / 20.7 (14.7 / 16.5 / 19.2), 17 MB 9.0 / 10.5 / 12.7 (8.2 / 9.3 / 10.8).
  const bool wide = !w16 && cx.w8a16_wide != 0 && n % 16 == 0 && ((uintptr_t)wq0 | (uintptr_t)wq1) % 16 == 0 &&
                    (cx.w8a16_wide == 2 || k * n * n_mats >= (int64_t)80 * 1000 * 1000);
  const int cols = wide ? 16 : 8, slab = 16 * cols;
  p.slabs = (int)((n + slab - 1) / slab);
  p.ks = (int)((k + kStep - 1) / kStep);
  const int64_t slabs_total = (int64_t)p.slabs * n_mats, units = slabs_total * p.ks;
  int64_t wgs = skinny_workgroups(slabs_total, p.ks, std::max<int64_t>(1, cx.w8a16_wgs_per_cu * cx.num_cu), cx.w8a16_min_steps);
  // (units * wgs is computed in 32 bits by the kernels; shapes beyond that get a workgroup per slab)
  const bool mapped = units * wgs < (1ll << 31);
  if (!mapped) wgs = slabs_total;
  p.per_wg = (int)(units / wgs);
  p.extra = (int)(units % wgs);
  p.mapped = mapped ? 1 : 0;
  out->map = mapped ? SlabMap{(unsigned)units, (unsigned)wgs, (unsigned)p.ks, wide ? 8 : 7, p.slabs} : SlabMap{};
  out->splits = mapped ? (int)((p.ks * wgs + units - 1) / units) + 1 : 1;  // at most
  // scratch for 32 rows whatever m: a call sized once fits every smaller and larger batch of the shape, also under capture
  const size_t one = (size_t)out->splits * kMaxM * n * sizeof(float);
  void* ws = nullptr;
  int rc = workspace(one * n_mats, &ws);
  if (rc) return rc;
  p.part[0] = reinterpret_cast<float*>(ws);
  p.part[1] = reinterpret_cast<float*>(reinterpret_cast<char*>(ws) + one);
  const bool bf = x_dtype == PTO_HIP_BF16, nt = cx.w8a16_nt != 0, two = m > 16;
  auto go = [&](auto w8, auto kcols) {
    constexpr bool W8 = decltype(w8)::value;
    constexpr int C = decltype(kcols)::value;
    if (bf) return two ? launch_partial<true, W8, C, 2>(p, (int)wgs, nt, st) : launch_partial<true, W8, C, 1>(p, (int)wgs, nt, st);
    return two ? launch_partial<false, W8, C, 2>(p, (int)wgs, nt, st) : launch_partial<false, W8, C, 1>(p, (int)wgs, nt, st);
  };
  typedef std::integral_constant<int, 8> C8;
  typedef std::integral_constant<int, 16> C16;
  rc = w16 ? go(std::false_type{}, C8{}) : wide ? go(std::true_type{}, C16{}) : go(std::true_type{}, C8{});
  if (rc) return rc;
  out->part[0] = p.part[0];
  out->part[1] = wq1 ? p.part[1] : nullptr;
  out->slab_stride = m * n;
  out->scaled = false;
  return PTO_HIP_OK;
}

int w8a16_finish(const W8Partials& parts, const float* scale0, const float* scale1, const void* residual,
                 int res_dtype, void* out, int out_dtype, bool out_blocked, int64_t m, int64_t n, hipStream_t st) {
  FinishParams f{};
  f.part0 = parts.part[0];
  f.part1 = parts.part[1];
  f.scale0 = scale0;
  f.scale1 = scale1;
  f.residual = residual;
  f.out = out;
  f.m = (int)m;
  f.n = (int)n;
  f.splits = parts.splits;
  f.res_dtype = res_dtype;
  f.out_dtype = out_dtype;
  f.out_blocked = out_blocked ? 1 : 0;
  f.stride = parts.slab_stride;
  f.map = parts.map;
  hipLaunchKernelGGL(w8a16_finish_kernel, dim3((unsigned)((n / 4 + 255) / 256), (unsigned)m), dim3(256), 0, st, f);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

bool w8a16_finish_norm_fits(int64_t n) { return n % 4 == 0 && n <= 4 * kNormThreads * kNormVec; }

int w8a16_finish_norm(const W8Partials& parts, const float* scale, const void* residual, int res_dtype,
                      float* sum_out, const float* gamma, void* normed_out, int out_dtype, bool out_blocked,
                      int64_t m, int64_t n, float eps, hipStream_t st) {
  FinishNormParams f{};
  f.part = parts.part[0];
  f.scale = scale;
  f.residual = residual;
  f.sum_out = sum_out;
  f.gamma = gamma;
  f.normed_out = normed_out;
  f.n = (int)n;
  f.splits = parts.splits;
  f.res_dtype = res_dtype;
  f.out_dtype = out_dtype;
  f.out_blocked = out_blocked ? 1 : 0;
  f.eps = eps;
  f.stride = parts.slab_stride;
  f.map = parts.map;
  hipLaunchKernelGGL(w8a16_finish_norm_kernel, dim3((unsigned)m), dim3(kNormThreads), 0, st, f);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

}  // namespace pto_hip

extern "C" int pto_hip_w8a16_matmul(const void* x, const void* w_q, const float* w_scale,
                                    const void* residual, void* out, int64_t m, int64_t k, int64_t n,
                                    int x_dtype, int res_dtype, int out_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  int rc = check_common("w8a16_matmul", m, k, n, x_dtype, out_dtype);
  if (rc) return rc;
  if (m == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(x && w_q && w_scale && out, "w8a16_matmul: null tensor pointer");
  PTO_CHECK_ARG(((uintptr_t)x % 16 == 0) && ((uintptr_t)w_q % 8 == 0) && ((uintptr_t)w_scale % 16 == 0) &&
                    ((uintptr_t)out % 16 == 0) && ((uintptr_t)residual % 16 == 0),
                "w8a16_matmul: misaligned operand");
  if (residual)
    PTO_CHECK_ARG(res_dtype == PTO_HIP_FP32 || res_dtype == PTO_HIP_BF16 || res_dtype == PTO_HIP_FP16,
                  "w8a16_matmul: residual dtype %s not in {FP32, BF16, FP16}", dtype_name(res_dtype));
  hipStream_t st = (hipStream_t)stream;
  // Many rows: one tiled GEMM that reads the codes once.
  if (gemm_w8_fits(x, w_q, nullptr, residual, out, m, k, n, x_dtype, out_dtype))
    return gemm_w8(x, w_q, w_scale, nullptr, nullptr, residual, res_dtype, out, m, k, n, x_dtype, out_dtype, st);
  // The kernel holds 32 rows of x per pass; more rows stream the weights once per pass, in order
  // on the stream (the partial buffer is reused).
  for (int64_t r0 = 0; r0 < m; r0 += kMaxM) {
    const int64_t rows = std::min<int64_t>(kMaxM, m - r0);
    W8Partials parts{};
    rc = w8a16_partials(byte_offset(x, r0 * k * 2), false, w_q, nullptr, rows, k, n, x_dtype, st, &parts);
    if (rc) return rc;
    rc = w8a16_finish(parts, w_scale, nullptr,
                      residual ? byte_offset(residual, r0 * n * dtype_bytes(res_dtype)) : nullptr, res_dtype,
                      byte_offset(out, r0 * n * dtype_bytes(out_dtype)), out_dtype, false, rows, n, st);
    if (rc) return rc;
  }
  return PTO_HIP_OK;
}

extern "C" int pto_hip_w8a16_swiglu(const void* x, const void* wg_q, const float* wg_scale,
                                    const void* wu_q, const float* wu_scale, void* out, int64_t m,
                                    int64_t k, int64_t n, int x_dtype, int out_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  int rc = check_common("w8a16_swiglu", m, k, n, x_dtype, out_dtype);
  if (rc) return rc;
  if (m == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(x && wg_q && wg_scale && wu_q && wu_scale && out, "w8a16_swiglu: null tensor pointer");
  PTO_CHECK_ARG(((uintptr_t)x % 16 == 0) && ((uintptr_t)wg_q % 8 == 0) && ((uintptr_t)wu_q % 8 == 0) &&
                    ((uintptr_t)wg_scale % 16 == 0) && ((uintptr_t)wu_scale % 16 == 0) && ((uintptr_t)out % 16 == 0),
                "w8a16_swiglu: misaligned operand");
  hipStream_t st = (hipStream_t)stream;
  if (gemm_w8_fits(x, wg_q, wu_q, nullptr, out, m, k, n, x_dtype, out_dtype))
    return gemm_w8(x, wg_q, wg_scale, wu_q, wu_scale, nullptr, 0, out, m, k, n, x_dtype, out_dtype, st);
  for (int64_t r0 = 0; r0 < m; r0 += kMaxM) {  // 32 rows per pass, as in w8a16_matmul
    const int64_t rows = std::min<int64_t>(kMaxM, m - r0);
    W8Partials parts{};
    rc = w8a16_partials(byte_offset(x, r0 * k * 2), false, wg_q, wu_q, rows, k, n, x_dtype, st, &parts);
    if (rc) return rc;
    rc = w8a16_finish(parts, wg_scale, wu_scale, nullptr, 0, byte_offset(out, r0 * n * dtype_bytes(out_dtype)),
                      out_dtype, false, rows, n, st);
    if (rc) return rc;
  }
  return PTO_HIP_OK;
}

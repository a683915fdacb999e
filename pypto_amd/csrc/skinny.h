// Kernels of the skinny projections (w8a16.hip): the partial-sum kernel, and the form of it for up to four rows that makes its
// activations itself.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "attn_merge.h"
#include "common.h"
#include "slab_sum.h"

namespace pto_hip {
namespace skinny {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;

constexpr int kStep = 32;                // k rows per step
constexpr int kMaxM = kW8MaxM;
constexpr int kFusedLds = 160 * 1024;   // most LDS of the fused form
constexpr int kWaves = 4;                // wavefronts per workgroup of the partial kernel

constexpr int kMaxFusedRows = kSkinnyFusedRows;
constexpr int kNormOwn = 2;      // 8-row pieces of its share a thread normalises at most
constexpr int kSwigluQuads = 2;  // quads of SwiGLU outputs a thread holds the slabs of at once
constexpr int kNormVecs = 4;  // 16-byte pieces of a row that a thread of the RMSNorm kernels holds at most

// What a workgroup multiplies: activations that a launch before it wrote, or ones that it makes itself, in LDS, of the k rows
// of its share - the launch that would have written them falls away (skinny_fuses has the rule).
enum Source {
  kGiven = 0,
  kNorm = 1,      // RMSNorm of x, as rms_norm_vec_kernel computes it
  kSwiglu = 2,    // SiLU(gate) * up of the pair in front, as w8a16_finish_kernel computes it
  kMerge128 = 3,  // attention partials merged, as attn_reduce_kernel does, at head_dim 128
  kMerge256 = 4,  // ... and 256
};

struct GemvParams {
  const uint16_t* x;    // [M, K] 16-bit activations
  const void* wq[2];    // [K, N] each (int8 codes or 16-bit weights); the second is the up projection of a pair
  float* part[2];       // [partial slabs, M, N] each
  int m, k, n, x_blocked;  // x_blocked: activations stored [K/8][32][8] (see w8a16_partials) instead of row-major
  int slabs, ks;        // output slabs of one matrix, 32-row steps of one slab
  int per_wg, extra;    // units / workgroups and its remainder (see SlabMap)
  int mapped;           // 0: a workgroup per slab
  int per_slab;         // workgroups of a slab (fused form)
  int wgs;              // workgroups; gridDim.x lies behind src, two lines of arguments further (0.03 us a launch)
  ProjectionSource src; // unless kGiven
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

// acc += activations x one stage of weights: 8 k rows of kCols channels a lane, transposed in registers into MFMA operands.
// keep false: rows that a last step repeats, zero in both operands - an infinite 16-bit weight there must not become a NaN.  They
// are cleared by the transposing v_perm_b32 itself (selector 12 gives a zero byte): behind a branch of their own in the last step layers of one
// to four rows were 0.2 us slower, and the 32-row form took 280 registers instead of 256.
template <bool BF16, bool W8, int kCols, int MT, typename W>
__device__ __forceinline__ void multiply(const W (&w)[8], const u32x4 (&x)[MT], bool keep, f32x4 (&acc)[kCols][MT]) {
  const uint32_t even = keep ? 0x05040100u : 0x0c0c0c0cu, odd = keep ? 0x07060302u : 0x0c0c0c0cu;
  u32x4 a[MT];
#pragma unroll
  for (int h = 0; h < MT; ++h) a[h] = keep ? x[h] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < kCols; ++i) {
    // channel n0 + i: its 8 k-values, as packed pairs (k, k+1)
    u32x4 b;
    if constexpr (W8) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t w0 = w[2 * q][i >> 2];
        const uint32_t w1 = w[2 * q + 1][i >> 2];
        const float f0 = (float)(int8_t)(w0 >> ((i & 3) * 8));
        const float f1 = (float)(int8_t)(w1 >> ((i & 3) * 8));
        b[q] = pack_pair<BF16>(f0, f1);
      }
    } else {
      // 16-bit weights: element i of rows 2q and 2q+1 (an 8x8 transpose in registers)
      const uint32_t sel = (i & 1) ? odd : even;
#pragma unroll
      for (int q = 0; q < 4; ++q) b[q] = __builtin_amdgcn_perm(w[2 * q + 1][i >> 1], w[2 * q][i >> 1], sel);
    }
#pragma unroll
    for (int h = 0; h < MT; ++h) acc[i][h] = mfma16<BF16>(a[h], b, acc[i][h]);
    __builtin_amdgcn_sched_barrier(0);  // keep the conversions next to their MFMAs
  }
}

// End of a run: the wavefronts' accumulators through LDS into partial slab `part` of the matrix's slab.  acc[i][h][r] is row
// h*16 + 4*kg + r, channel c*kCols + i; the float4s of a row are kept in the order (v, c) - channels c*kCols + 4v .. -
// so that neither the writes nor the reads of 16 lanes collide in a bank.
template <int kCols, int MT>
__device__ __forceinline__ void store_run(const GemvParams& p, float* red, const f32x4 (&acc)[kCols][MT], int tid, int mat, int slab, int part) {
  constexpr int kSlab = 16 * kCols, kRows = 16 * MT, kQuads = kSlab / 4;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, kg = lane >> 4;
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
  const int q = tid % kQuads, n = slab * kSlab + (q & 15) * kCols + (q >> 4) * 4;
  float* out = p.part[mat] + (size_t)part * p.m * p.n + n;
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
}

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
  const int wg = blockIdx.x, wgs = p.wgs;
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
  // cleared in the activations and in 16-bit weights.  A row address is a wavefront-uniform row base plus a
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
    multiply<BF16, W8, kCols, MT>(s.w, s.xa, k_ok, acc);
  };

  auto finish_run = [&](const Cursor& cur) {
    const int mat = cur.slab >= p.slabs ? 1 : 0;
    // partial slab number: how many workgroups before this one hold steps of the slab (the one
    // that holds its first unit has number 0)
    const int first = cur.slab * p.ks;
    const int owner = p.mapped ? (int)(((unsigned)(first + 1) * (unsigned)wgs - 1) / (unsigned)(p.per_wg * wgs + p.extra)) : wg;
    store_run<kCols, MT>(p, red, acc, tid, mat, cur.slab - mat * p.slabs, wg - owner);
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
  add_slabs(src, splits, stride, sum);
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

// SiLU(gate) * up of four channels of row m of a pair's partial slabs.
__device__ __forceinline__ float4 swiglu_quad(const float* part0, const float* part1, const float* scale0, const float* scale1,
                                              const SlabMap& map, int splits, size_t stride, int m, int n, int nn) {
  const int splits0 = slab_count(map, splits, 0, n), splits1 = slab_count(map, splits, 1, n);
  float4 a, u;
  if (splits0 == splits1) {
    const float* parts[2] = {part0, part1};
    const float* scales[2] = {scale0, scale1};
    f32x4 sum[2];
    sum_splits<2>(parts, scales, splits0, stride, m, n, nn, sum);
    a = float4{sum[0][0], sum[0][1], sum[0][2], sum[0][3]};
    u = float4{sum[1][0], sum[1][1], sum[1][2], sum[1][3]};
  } else {
    a = sum_splits(part0, scale0, splits0, stride, m, n, nn);
    u = sum_splits(part1, scale1, splits1, stride, m, n, nn);
  }
  return float4{silu_mul(a.x, u.x), silu_mul(a.y, u.y), silu_mul(a.z, u.z), silu_mul(a.w, u.w)};
}

// ---- activations made by the workgroup that multiplies them --------------------------------------
// Rows 0 .. m-1 of k [k_lo, k_hi) into LDS at xs, `pitch` elements apart: what a launch in front would have computed for these
// k rows, to the bit.  request() asks for all that fits the registers before the first weights are asked for - loads
// come back in order -, finish() computes; what does not fit is read there.
template <bool BF16, int SRC>
struct Activations;

// RMSNorm of x: every workgroup sums the squares of the whole row and normalises its own part.
template <bool BF16>
struct Activations<BF16, kNorm> {
  typedef typename std::conditional<BF16, __bf16, _Float16>::type T;
  typedef __attribute__((__vector_size__(8 * sizeof(T)))) T vec8;
  static constexpr int kThreads = kWaves * 64, kOwn = kNormOwn;  // pieces of 8 k rows of the own part a thread normalises
  vec8 v[kMaxFusedRows][kNormVecs], own[kMaxFusedRows][kOwn];
  float4 g0[kOwn], g1[kOwn];

  __device__ __forceinline__ void request(const GemvParams& p, int k_lo, int k_hi) {
    const int tid = threadIdx.x, last = p.k / 8 - 1, lo = k_lo / 8, hi = k_hi / 8;
#pragma unroll
    for (int m = 0; m < kMaxFusedRows; ++m) {
      if (m >= p.m) break;
      const vec8* xr = reinterpret_cast<const vec8*>(p.x + (size_t)m * p.k);
#pragma unroll
      for (int u = 0; u < kNormVecs; ++u)
        if (u * kThreads <= last) v[m][u] = xr[min(tid + u * kThreads, last)];
#pragma unroll
      for (int u = 0; u < kOwn; ++u)
        if (lo + u * kThreads < hi) own[m][u] = xr[min(lo + tid + u * kThreads, hi - 1)];
    }
#pragma unroll
    for (int u = 0; u < kOwn; ++u)
      if (lo + u * kThreads < hi) {
        const int i = min(lo + tid + u * kThreads, hi - 1);
        g0[u] = reinterpret_cast<const float4*>(p.src.gamma)[2 * i];
        g1[u] = reinterpret_cast<const float4*>(p.src.gamma)[2 * i + 1];
      }
  }
  __device__ __forceinline__ void finish(const GemvParams& p, uint16_t* xs, int pitch, int k_lo, int k_hi, float* scratch) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nvec = p.k / 8, pieces = (k_hi - k_lo) / 8;
#pragma unroll
    for (int m = 0; m < kMaxFusedRows; ++m) {
      if (m >= p.m) break;
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < kNormVecs; ++u)
        if (tid + u * kThreads < nvec) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float f = (float)v[m][u][e];
            ss += f * f;
          }
        }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
      if (lane == 0) scratch[m * kWaves + wave] = ss;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int m = 0; m < kMaxFusedRows; ++m) {
      if (m >= p.m) break;
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) tot += scratch[m * kWaves + w];
      const float inv = rsqrtf(tot / (float)p.k + p.src.eps);
#pragma unroll
      for (int u = 0; u < kOwn; ++u) {
        const int i = tid + u * kThreads;
        if (i < pieces) {
          const float g[8] = {g0[u].x, g0[u].y, g0[u].z, g0[u].w, g1[u].x, g1[u].y, g1[u].z, g1[u].w};
          vec8 o;
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = (T)((float)own[m][u][e] * inv * g[e]);
          *reinterpret_cast<vec8*>(reinterpret_cast<T*>(xs) + m * pitch + i * 8) = o;
        }
      }
    }
  }
};

// SiLU(gate) * up of the pair's partial slabs.
template <bool BF16>
struct Activations<BF16, kSwiglu> {
  typedef typename std::conditional<BF16, __bf16, _Float16>::type T;
  typedef __attribute__((__vector_size__(4 * sizeof(T)))) T vec4;
  static constexpr int kQuads = kSwigluQuads, kSlabs = 4;  // quads of a thread and slabs of a channel held at once
  f32x4 t[kQuads][2][kSlabs], scale[kQuads][2];

  __device__ __forceinline__ void request(const GemvParams& p, int k_lo, int k_hi) {
    const ProjectionSource& s = p.src;
    const int quads = (k_hi - k_lo) / 4;
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
      if (u * kWaves * 64 >= p.m * quads) break;
      const int i = min((int)threadIdx.x + u * kWaves * 64, p.m * quads - 1), m = i / quads, n = k_lo + 4 * (i - m * quads);
#pragma unroll
      for (int mat = 0; mat < 2; ++mat) {
        const float* src = s.pair.part[mat] + (size_t)m * p.k + n;
        const int last = slab_count(s.pair.map, s.pair.splits, mat, n) - 1;
        auto get = [&](int b) { t[u][mat][b] = *reinterpret_cast<const f32x4*>(src + (size_t)min(b, last) * s.pair.slab_stride); };
        get(0);
        get(1);
        if (s.pair.splits > 2) {  // (at most: shares that cross slabs give a slab of two shares' work three parts)
          get(2);
          get(3);
        }
        const float* sc = mat ? s.scale1 : s.scale0;
        scale[u][mat] = sc ? *reinterpret_cast<const f32x4*>(sc + n) : f32x4{1.f, 1.f, 1.f, 1.f};
      }
    }
  }
  __device__ __forceinline__ void finish(const GemvParams& p, uint16_t* xs, int pitch, int k_lo, int k_hi, float*) {
    const ProjectionSource& s = p.src;
    const int quads = (k_hi - k_lo) / 4;
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
      const int i = (int)threadIdx.x + u * kWaves * 64;
      if (i < p.m * quads) {
        const int m = i / quads, n = k_lo + 4 * (i - m * quads);
        f32x4 sum[2];
#pragma unroll
        for (int mat = 0; mat < 2; ++mat) {
          const int count = slab_count(s.pair.map, s.pair.splits, mat, n);
          sum[mat] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int b = 0; b < kSlabs; ++b)
            if (b < count) sum[mat] += t[u][mat][b];
          const float* src = s.pair.part[mat] + (size_t)m * p.k + n;
          for (int b = kSlabs; b < count; ++b) sum[mat] += *reinterpret_cast<const f32x4*>(src + (size_t)b * s.pair.slab_stride);
          sum[mat] *= scale[u][mat];
        }
        vec4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = (T)silu_mul(sum[0][e], sum[1][e]);
        *reinterpret_cast<vec4*>(reinterpret_cast<T*>(xs) + m * pitch + n - k_lo) = y;
      }
    }
  }
};

// Attention partials merged: a wavefront per (row, head) of the part, as merge_row sums them.
template <bool BF16, int D>
struct MergeActivations {
  typedef typename std::conditional<BF16, __bf16, _Float16>::type T;
  static constexpr int kHeld = kMergeHeld;  // partitions, D / 64 channels of each
  float2 own;
  float pv[kHeld][D / 64];
  int ctx, m, head;
  bool have;

  __device__ __forceinline__ void request(const GemvParams& p, int k_lo, int k_hi) {
    const AttnPartials& a = p.src.attn;
    const int lane = threadIdx.x & 63, i = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int head0 = k_lo / D, span = (k_hi - 1) / D + 1 - head0;
    have = i < p.m * span;
    if (!have) return;
    m = i / span;
    head = head0 + i - m * span;
    const size_t row = (size_t)m * (p.k / D) + head;
    ctx = a.ctx_lens[m];
    own = *reinterpret_cast<const float2*>(a.ml + (row * a.n_part + min(lane, a.n_part - 1)) * 2);
    const float* po = a.o + row * a.n_part * D + lane;
#pragma unroll
    for (int b = 0; b < kHeld; b += 8) {
      if (b >= a.n_part) break;
#pragma unroll
      for (int u = b; u < b + 8; ++u)
#pragma unroll
        for (int k = 0; k < D / 64; ++k) pv[u][k] = po[(size_t)min(u, a.n_part - 1) * D + k * 64];
    }
  }
  __device__ __forceinline__ void finish(const GemvParams& p, uint16_t* xs, int pitch, int k_lo, int k_hi, float*) {
    if (!have) return;
    const AttnPartials& a = p.src.attn;
    const int lane = threadIdx.x & 63;
    const int c = ctx < 0 ? 0 : (ctx > a.ctx_cap ? a.ctx_cap : ctx);
    const int np = (c + a.tpp - 1) / a.tpp;
    float o[D / 64], l = 0.f;
#pragma unroll
    for (int k = 0; k < D / 64; ++k) o[k] = 0.f;
    if (a.n_part <= attn::kReduceFast) {
      float mx = attn::kMinMax;
#pragma unroll
      for (int u = 0; u < attn::kReduceFast; ++u) mx = u < np ? fmaxf(mx, read(own.x, u)) : mx;
#pragma unroll
      for (int u = 0; u < attn::kReduceFast; ++u) {
        const float wgt = __builtin_amdgcn_exp2f(read(own.x, u) - mx);
        if (u < np) {
          l += wgt * read(own.y, u);
#pragma unroll
          for (int k = 0; k < D / 64; ++k) o[k] += wgt * pv[u][k];
        }
      }
    } else {
      float mx = lane < np ? own.x : attn::kMinMax;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
      const float wgt = lane < np ? __builtin_amdgcn_exp2f(own.x - mx) : 0.f;
      l = lane < np ? wgt * own.y : 0.f;
#pragma unroll
      for (int b = 0; b < kHeld; b += 8) {
        if (b >= np) break;
#pragma unroll
        for (int u = b; u < b + 8; ++u) {
          const float w = read(wgt, u);
#pragma unroll
          for (int k = 0; k < D / 64; ++k) o[k] = u < np ? o[k] + w * pv[u][k] : o[k];
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int k = 0; k < D / 64; ++k) {
      const int kk = head * D + k * 64 + lane;
      // Rounded to fp32 first, as the merge launch writes it: left to itself the compiler makes product and cast one v_fma_mixlo_f16, which
      // rounds once, and a call then differed from the measured ones of its signature, which merge in a launch.
      float y = o[k] * inv;
      asm("" : "+v"(y));
      if (kk >= k_lo && kk < k_hi) reinterpret_cast<T*>(xs)[m * pitch + kk - k_lo] = (T)y;
    }
  }
  static __device__ __forceinline__ float read(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
  }
};
template <bool BF16>
struct Activations<BF16, kMerge128> : MergeActivations<BF16, 128> {};
template <bool BF16>
struct Activations<BF16, kMerge256> : MergeActivations<BF16, 256> {};

// The partial kernel for up to kMaxFusedRows rows and shares that lie in one slab (skinny_fuses).  The first two rounds of
// weights are requested before the activations are made, so most of what that takes passes while they are on their way.
template <bool BF16, bool W8, int kCols, int SRC>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 2))) void skinny_fused_kernel(GemvParams p) {
  constexpr int kSlab = 16 * kCols;
  constexpr int kWBytes = W8 ? 1 : 2;
  typedef typename std::conditional<(W8 && kCols == 8), u32x2, u32x4>::type wvec_t;
  extern __shared__ __attribute__((aligned(16))) float red[];  // [kWaves][16][kSlab], then the activations
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int slab = blockIdx.x / p.per_slab, part = blockIdx.x - slab * p.per_slab;
  // (as the plain kernel's units fall: workgroup w's first is w * units / workgroups, here slab * ks + part * ks / per_slab)
  const int s0 = part * p.ks / p.per_slab, s1 = (part + 1) * p.ks / p.per_slab;
  const int rounds = (s1 - s0 + kWaves - 1) / kWaves;
  const int k_lo = min(s0 * kStep, p.k - kStep), k_hi = min(s1 * kStep, p.k), pitch = k_hi - k_lo + 8;
  uint16_t* const xs = reinterpret_cast<uint16_t*>(red + kWaves * 16 * kSlab);
  const int mat = slab >= p.slabs ? 1 : 0;
  const int n0 = min((slab - mat * p.slabs) * kSlab + c * kCols, p.n - kCols);
  const size_t lane_off = ((size_t)n0 + (size_t)(kg * 8) * p.n) * kWBytes;
  const char* const wmat = reinterpret_cast<const char*>(p.wq[mat]);

  auto row_of = [&](int round) { return min(min(s0 + round * kWaves + wave, s1 - 1) * kStep, p.k - kStep); };
  auto load = [&](wvec_t (&w)[8], int round) {
    const char* wbase = wmat + (size_t)row_of(round) * p.n * kWBytes;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      w[e] = __builtin_nontemporal_load(reinterpret_cast<const wvec_t*>(wbase + (size_t)e * p.n * kWBytes + lane_off));
  };
  f32x4 acc[kCols][1];
#pragma unroll
  for (int i = 0; i < kCols; ++i) acc[i][0] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const wvec_t (&w)[8], int round) {
    const int step = s0 + round * kWaves + wave;
    if (step >= s1) return;  // uniform
    const int k = row_of(round) + kg * 8;
    const u32x4 act = *reinterpret_cast<const u32x4*>(xs + min(c, p.m - 1) * pitch + k - k_lo);
    const u32x4 a[1] = {act};
    multiply<BF16, W8, kCols, 1>(w, a, k >= step * kStep, acc);
  };

  wvec_t w0[8], w1[8];
  Activations<BF16, SRC> x;
  x.request(p, k_lo, k_hi);
  __builtin_amdgcn_sched_barrier(0);
  load(w0, 0);
  load(w1, 1);
  __builtin_amdgcn_sched_barrier(0);
  x.finish(p, xs, pitch, k_lo, k_hi, red);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  int r = 0;
  for (; r + 3 < rounds; r += 2) {
    compute(w0, r);
    load(w0, r + 2);
    compute(w1, r + 1);
    load(w1, r + 3);
  }
  compute(w0, r);
  if (r + 2 < rounds) {
    load(w0, r + 2);
    compute(w1, r + 1);
    compute(w0, r + 2);
  } else if (r + 1 < rounds) {
    compute(w1, r + 1);
  }
  store_run<kCols, 1>(p, red, acc, tid, mat, slab - mat * p.slabs, part);
}

template <bool BF16, bool W8, int kCols, int SRC>
int launch_fused(const GemvParams& p, int wgs, size_t smem, hipStream_t st) {
  auto kern = skinny_fused_kernel<BF16, W8, kCols, SRC>;
  static std::atomic<bool> attr_set{false};  // per instantiation; callers hold the dispatch lock
  if (!attr_set.load(std::memory_order_acquire)) {
    PTO_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kFusedLds));
    attr_set.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(kWaves * 64), smem, st, p);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}
template <int SRC>
int launch_fused_source(const GemvParams& p, bool bf16, bool w16, bool wide, int wgs, size_t smem, hipStream_t st) {
  if (w16) return bf16 ? launch_fused<true, false, 8, SRC>(p, wgs, smem, st) : launch_fused<false, false, 8, SRC>(p, wgs, smem, st);
  if (wide) return bf16 ? launch_fused<true, true, 16, SRC>(p, wgs, smem, st) : launch_fused<false, true, 16, SRC>(p, wgs, smem, st);
  return bf16 ? launch_fused<true, true, 8, SRC>(p, wgs, smem, st) : launch_fused<false, true, 8, SRC>(p, wgs, smem, st);
}

}  // namespace skinny
}  // namespace pto_hip

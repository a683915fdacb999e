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
#include "skinny.h"

namespace {

using namespace pto_hip::skinny;
using pto_hip::SlabMap;
using pto_hip::slab_count;

struct FinishParams {
  const float* part0;   // [splits, 32 or M, N]: `stride` elements between splits
  const float* part1;   // second projection for SwiGLU, or null
  const float* scale0;  // [N]
  const float* scale1;
  const void* residual; // [M, N] in res_dtype, or null
  void* out;            // [M, N]
  int m, n, splits, res_dtype, out_dtype;
  int out_rows;  // write out as [N/8][out_rows][8] for the next projection; 0: row-major
  int64_t stride;
  SlabMap map;
};

// Element index of (row m, channel n) in the blocked activation layout [N/8][rows][8].
__device__ __forceinline__ size_t blocked_index(int rows, int m, int n) { return ((size_t)(n >> 3) * rows + m) * 8 + (n & 7); }

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

// BLOCKED: eight rows and 128 channels a workgroup, a wavefront's 64 quads whole 128-byte lines of the blocked layout (8 rows x 8
// channels); rows of the layout written one a workgroup, its lines are put together from eight XCDs' caches.  For the rows that a layer streams
// (33 to 96); up to 32 the row form is as fast (16 rows x 17408 4.8 us either way) or faster (7 x 2752 3.4 against 4.2).
template <bool BLOCKED>
__global__ __launch_bounds__(256) void w8a16_finish_kernel(FinishParams p) {
  const int n = BLOCKED ? blockIdx.x * 128 + (threadIdx.x >> 3) * 4 : (blockIdx.x * 256 + threadIdx.x) * 4;
  const int m = BLOCKED ? blockIdx.y * 8 + (threadIdx.x & 7) : blockIdx.y;
  if (n >= p.n || (BLOCKED && m >= p.m)) return;
  const size_t idx = (size_t)m * p.n + n;
  float4 r = {0.f, 0.f, 0.f, 0.f};  // requested with the slabs
  if (p.residual) r = load4_as_f32(p.residual, idx, p.res_dtype);
  float4 a;
  if (p.part1) {
    a = swiglu_quad(p.part0, p.part1, p.scale0, p.scale1, p.map, p.splits, (size_t)p.stride, m, n, p.n);
  } else {
    a = sum_splits(p.part0, p.scale0, slab_count(p.map, p.splits, 0, n), (size_t)p.stride, m, n, p.n);
  }
  if (p.residual) {
    a.x += r.x; a.y += r.y; a.z += r.z; a.w += r.w;
  }
  store4_from_f32(p.out, p.out_rows ? blocked_index(p.out_rows, m, n) : idx, p.out_dtype, a);
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
  int out_rows;
  int spread_rows;  // see blocked_row
  float eps;
  int64_t stride;  // elements between splits
  SlabMap map;
};

__global__ __launch_bounds__(kNormThreads) void w8a16_finish_norm_kernel(FinishNormParams p) {
  const int m = pto_hip::blocked_row(blockIdx.x, p.spread_rows);
  float4 v[kNormVec];
  float4 g[kNormVec];  // requested with the row, so that the second pass waits for nothing
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < kNormVec; ++u) {
    const int n = (threadIdx.x + u * kNormThreads) * 4;
    if (n < p.n) {
      g[u] = *reinterpret_cast<const float4*>(p.gamma + n);
      const float4 r = load4_as_f32(p.residual, (size_t)m * p.n + n, p.res_dtype);
      float4 a = sum_splits(p.part, p.scale, slab_count(p.map, p.splits, 0, n), (size_t)p.stride, m, n, p.n);
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
      store4_from_f32(p.normed_out, p.out_rows ? blocked_index(p.out_rows, m, n) : (size_t)m * p.n + n, p.out_dtype, y);
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

int skinny_norm_launch(const skinny::GemvParams& p, bool bf16, bool w16, bool wide, int wgs, size_t smem, hipStream_t st);
int skinny_swiglu_launch(const skinny::GemvParams& p, bool bf16, bool w16, bool wide, int wgs, size_t smem, hipStream_t st);
int skinny_merge_launch(const skinny::GemvParams& p, bool bf16, bool w16, bool wide, int wgs, size_t smem, hipStream_t st);

namespace {
// How a projection's units fall to workgroups.
struct SkinnyPlan {
  bool wide, mapped;
  int cols, slabs, ks, splits, per_slab;  // per_slab: workgroups of every slab; 0: shares cross slabs
  int64_t units, wgs;
};
SkinnyPlan plan_skinny(int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16) {
  const Context& cx = ctx();
  const int n_mats = wq1 ? 2 : 1;
  SkinnyPlan q{};
  // int8 codes are read 16 per lane (256-channel slabs, 256-byte row pieces instead of 128) when rows and base
  // addresses allow 16-byte loads and the matrices are large.  Twice the channels in a slab are twice the partial
  // sums at the same number of workgroups, and 32 instead of 16 KB per wavefront through LDS at the end of a run.
  // Measured with their finish at 1 / 16 / 32 rows: 178 MB 36.0 / 38.8 / 44.6 us (8 per lane: 36.4 / 42.0 / 50.2), 117 MB
  // 24.1 / 26.0 / 29.6 (25.6 / 29.2 / 34.0), 89 MB 20.4 / 22.1 / 25.7 (21.9 / 24.9 / 28.6); but 67 MB 16.5 / 18.2 / 21.7
  // (15.6 / 17.7 / 20.7), 59 MB 15.8 / 17.5 / 20.7 (14.7 / 16.5 / 19.2), 17 MB 9.0 / 10.5 / 12.7 (8.2 / 9.3 / 10.8).
  q.wide = !w16 && cx.w8a16_wide != 0 && n % 16 == 0 && ((uintptr_t)wq0 | (uintptr_t)wq1) % 16 == 0 &&
           (cx.w8a16_wide == 2 || k * n * n_mats >= (int64_t)80 * 1000 * 1000);
  q.cols = q.wide ? 16 : 8;
  const int slab = 16 * q.cols;
  q.slabs = (int)((n + slab - 1) / slab);
  q.ks = (int)((k + kStep - 1) / kStep);
  const int64_t slabs_total = (int64_t)q.slabs * n_mats;
  q.units = slabs_total * q.ks;
  q.wgs = skinny_workgroups(slabs_total, q.ks, std::max<int64_t>(1, cx.w8a16_wgs_per_cu * cx.num_cu), cx.w8a16_min_steps);
  // (units * wgs is computed in 32 bits by the kernels; shapes beyond that get a workgroup per slab)
  q.mapped = q.units * q.wgs < (1ll << 31);
  if (!q.mapped) q.wgs = slabs_total;
  q.per_slab = q.wgs % slabs_total == 0 && q.wgs / slabs_total <= q.ks ? (int)(q.wgs / slabs_total) : 0;
  // at most; whole shares are as many for every slab
  q.splits = q.per_slab ? q.per_slab : (int)((q.ks * q.wgs + q.units - 1) / q.units) + 1;
  return q;
}
// LDS of the fused form: the sums and m rows of a share.
size_t fused_lds(const SkinnyPlan& q, int64_t m) {
  const size_t span = ((size_t)q.ks + q.per_slab - 1) / q.per_slab * kStep + kStep;
  return (size_t)kWaves * 16 * 16 * q.cols * sizeof(float) + (size_t)m * (span + 8) * 2;
}
}  // namespace

// The launch saved is 2 to 5 us of a chain of ten; what is made instead is made by every workgroup, so it pays while a thread's part is
// held in registers at once, one round trip to the caches (decoder layer, us, one / two rows, separate launch -> made here):
// kNorm, up to 4 rows: 4096 wide int8 71.9 / 75.1 -> 70.4 / 73.1, 2048 wide 48.5 / 49.9 -> 46.8 / 48.3.
// kSwiglu, up to two quads of channels a thread, 2048 values a share: 5632 -> 2048 channels (352 k rows a share) 48.5 / 49.9 -> 46.9 / 48.6; 14336 -> 4096
// (1792) for one row 67.8 -> 66.9, 16-bit 98.1 -> 97.8, block of one token 64.2 -> 63.8; but 75.1 -> 76.7 for two rows, in two round trips;
// 20032 -> 8192 (5008) 142.9 -> 144.0.
// kMerge: a head a wavefront (32 heads, 4096 wide) 71.9 -> 69.7, two 75.1 -> 75.0, three (40 heads, 8192 wide) 142.9 -> 145.4.  More than the
// kMergeHeld partitions of a row keep their merge launch: 63 of them, in a loop past those held, 38.3 -> 42.6.
bool skinny_fuses(ProjectionSource::Kind kind, int64_t m, int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16, int64_t head_dim) {
  const Context& cx = ctx();
  if (!(cx.skinny_fuse >> (kind - 1) & 1) || cx.w8a16_nt == 0 || m > kSkinnyFusedRows || k % 16 != 0 || k < kStep) return false;
  const SkinnyPlan q = plan_skinny(k, n, wq0, wq1, w16);
  if (q.per_slab == 0 || fused_lds(q, m) > (size_t)kFusedLds) return false;
  const int64_t share = ((int64_t)q.ks + q.per_slab - 1) / q.per_slab * kStep;
  switch (kind) {
    case ProjectionSource::kNorm: return k <= 8 * 256 * kNormVecs && share + (k % kStep ? kStep : 0) <= 8 * 256 * kNormOwn;
    case ProjectionSource::kSwiglu: return m * share <= kSwigluQuads * 4 * kWaves * 64;
    case ProjectionSource::kMerge: {
      const bool whole = q.ks % q.per_slab == 0 && share % head_dim == 0;
      return m * (whole ? share / head_dim : share / head_dim + 2) <= kWaves;
    }
    default: return false;
  }
}

size_t skinny_fused_bytes(int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16) {
  const SkinnyPlan q = plan_skinny(k, n, wq0, wq1, w16);
  return (size_t)q.splits * kSkinnyFusedRows * n * sizeof(float) * (wq1 ? 2 : 1);
}

int w8a16_partials(const void* x, bool x_blocked, const void* wq0, const void* wq1, int64_t m, int64_t k, int64_t n,
                   int x_dtype, hipStream_t st, W8Partials* out, bool w16, const ProjectionSource* src, float* area) {
  const SkinnyPlan q = plan_skinny(k, n, wq0, wq1, w16);
  GemvParams p{};
  p.x = reinterpret_cast<const uint16_t*>(x);
  p.wq[0] = wq0;
  p.wq[1] = wq1;
  p.m = (int)m;
  p.k = (int)k;
  p.n = (int)n;
  p.x_blocked = x_blocked ? 1 : 0;
  p.slabs = q.slabs;
  p.ks = q.ks;
  p.per_wg = (int)(q.units / q.wgs);
  p.extra = (int)(q.units % q.wgs);
  p.mapped = q.mapped ? 1 : 0;
  p.per_slab = q.per_slab;
  p.wgs = (int)q.wgs;
  out->map = q.mapped ? SlabMap{(unsigned)q.units, (unsigned)q.wgs, (unsigned)q.ks, q.wide ? 8 : 7, q.slabs} : SlabMap{};
  out->splits = q.splits;
  // scratch for 32 rows whatever m: a call sized once fits every smaller and larger batch of the shape, also under capture
  size_t one = (size_t)q.splits * kMaxM * n * sizeof(float);
  int rc = PTO_HIP_OK;
  if (area) {
    one = (size_t)q.splits * kSkinnyFusedRows * n * sizeof(float);
  } else {
    void* ws = nullptr;
    if ((rc = workspace(one * (wq1 ? 2 : 1), &ws))) return rc;
    area = reinterpret_cast<float*>(ws);
  }
  p.part[0] = area;
  p.part[1] = reinterpret_cast<float*>(reinterpret_cast<char*>(area) + one);
  const Context& cx = ctx();
  const bool bf = x_dtype == PTO_HIP_BF16, nt = cx.w8a16_nt != 0, two = m > 16;
  const int wgs = (int)q.wgs;
  if (src && src->kind != ProjectionSource::kTensor) {
    p.src = *src;
    ctx().skinny_fused |= 1 << (src->kind - 1);
    const size_t smem = fused_lds(q, m);
    rc = src->kind == ProjectionSource::kNorm     ? skinny_norm_launch(p, bf, w16, q.wide, wgs, smem, st)
         : src->kind == ProjectionSource::kSwiglu ? skinny_swiglu_launch(p, bf, w16, q.wide, wgs, smem, st)
                                                  : skinny_merge_launch(p, bf, w16, q.wide, wgs, smem, st);
  } else {
    auto go = [&](auto w8, auto kcols) {
      constexpr bool W8 = decltype(w8)::value;
      constexpr int C = decltype(kcols)::value;
      if (bf) return two ? launch_partial<true, W8, C, 2>(p, wgs, nt, st) : launch_partial<true, W8, C, 1>(p, wgs, nt, st);
      return two ? launch_partial<false, W8, C, 2>(p, wgs, nt, st) : launch_partial<false, W8, C, 1>(p, wgs, nt, st);
    };
    typedef std::integral_constant<int, 8> C8;
    typedef std::integral_constant<int, 16> C16;
    rc = w16 ? go(std::false_type{}, C8{}) : q.wide ? go(std::true_type{}, C16{}) : go(std::true_type{}, C8{});
  }
  if (rc) return rc;
  out->part[0] = p.part[0];
  out->part[1] = wq1 ? p.part[1] : nullptr;
  out->slab_stride = m * n;
  out->scaled = false;
  return PTO_HIP_OK;
}

int w8a16_finish(const W8Partials& parts, const float* scale0, const float* scale1, const void* residual,
                 int res_dtype, void* out, int out_dtype, int out_rows, int64_t m, int64_t n, hipStream_t st) {
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
  f.out_rows = out_rows;
  f.stride = parts.slab_stride;
  f.map = parts.map;
  if (out_rows && m > kW8MaxM)
    hipLaunchKernelGGL(w8a16_finish_kernel<true>, dim3((unsigned)((n + 127) / 128), (unsigned)((m + 7) / 8)), dim3(256), 0, st, f);
  else
    hipLaunchKernelGGL(w8a16_finish_kernel<false>, dim3((unsigned)((n / 4 + 255) / 256), (unsigned)m), dim3(256), 0, st, f);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

bool w8a16_finish_norm_fits(int64_t n) { return n % 4 == 0 && n <= 4 * kNormThreads * kNormVec; }

int w8a16_finish_norm(const W8Partials& parts, const float* scale, const void* residual, int res_dtype,
                      float* sum_out, const float* gamma, void* normed_out, int out_dtype, int out_rows,
                      int64_t m, int64_t n, float eps, hipStream_t st) {
  FinishNormParams f{};
  f.part = parts.part[0];
  f.scale = scale;
  f.residual = residual;
  f.sum_out = sum_out;
  f.gamma = gamma;
  f.normed_out = normed_out;
  f.spread_rows = out_rows && m > kW8MaxM ? (int)m : 0;
  f.n = (int)n;
  f.splits = parts.splits;
  f.res_dtype = res_dtype;
  f.out_dtype = out_dtype;
  f.out_rows = out_rows;
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
                      byte_offset(out, r0 * n * dtype_bytes(out_dtype)), out_dtype, 0, rows, n, st);
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
                      out_dtype, 0, rows, n, st);
    if (rc) return rc;
  }
  return PTO_HIP_OK;
}

// Shared host-side plumbing of libpto_hip: status/error handling, the per-process
// context (device, workspace, options) and small dtype helpers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "pto_hip.h"

namespace pto_hip {

// Last failure message of the calling thread (pto_hip_last_error()).
std::string& last_error();
int fail(int status, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define PTO_CHECK_ARG(cond, ...)                                         \
  do {                                                                   \
    if (!(cond)) return ::pto_hip::fail(PTO_HIP_ERR_INVALID_VALUE, __VA_ARGS__); \
  } while (0)

#define PTO_CHECK_HIP(expr)                                                              \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess)                                                                \
      return ::pto_hip::fail(PTO_HIP_ERR_RUNTIME, "%s failed: %s (%s:%d)", #expr,        \
                             hipGetErrorString(_e), __FILE__, __LINE__);                 \
  } while (0)

// Process-wide state created by pto_hip_init().  One device per process, as one
// reference Worker is bound to one (platform, device) pair.
struct Context {
  bool initialized = false;
  int refcount = 0;  // pto_hip_init calls not yet matched by pto_hip_close
  int device = -1;
  int num_cu = 0;
  // Grow-only device scratch for partial results (attention partitions, FFN intermediates).
  void* workspace = nullptr;
  size_t workspace_bytes = 0;
  // Intermediates of the composed decoder layer (grow-only).
  void* layer_ws = nullptr;
  size_t layer_ws_bytes = 0;
  // Split-K slabs of the tiled GEMM (grow-only), apart from the two above so that a caller's
  // intermediates in either of them survive a GEMM launch.
  void* gemm_ws = nullptr;
  size_t gemm_ws_bytes = 0;
  // Buffers the scratch areas outgrew.  They stay allocated until pto_hip_close: launches
  // recorded into a HIP graph keep the address they were recorded with.
  std::vector<void*> retired;
  // 256 bytes of device flags written by kernels that report bad indices to the host.
  int* flags = nullptr;
  // options
  int64_t attn_tokens_per_partition = 0;
  int64_t attn_waves_per_cu = 0;
  int64_t attn_variant = -1;  // -1 by launch size, 0 partition grid, 1 evenly split form, 2 workgroup form (merge in LDS)
  // "attn_kernel_timing": the streaming attention kernel of every launch is bracketed by a pair of
  // HIP events on its stream; "attn_kernel_time_ns" reads the mean interval and drops the pairs.
  int64_t attn_kernel_timing = 0;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> attn_timed;
  int64_t attn_group_tiles = 0;  // cap on the query tiles one wavefront carries (0 = by group size)
  int64_t attn_autotune = 1;     // first calls of a launch signature time bit-identical launch shapes and keep the fastest
  int64_t attn_lean_siblings = 1;  // evenly split form: query tiles of one KV head on sibling wavefronts of one workgroup
  int64_t w8a16_nt = 1;            // skinny projections: weight rows read with non-temporal loads
  int64_t gemm_variant = 0;
  int64_t gemm_quad_rows = 0;    // tile height of the four-wavefront form: 0 = by estimate
  int64_t gemm_narrow = 0;       // small-call form of products with 16-bit or e4m3 weights: -1 never, 0 by estimate, 1..4 its tile
  int64_t gemm_splits = 0;       // k splits of the tiled GEMM: 0 = by shape, 1..16 = as given (when k allows)
  int64_t w8a16_wgs_per_cu = 1;  // most workgroups of the skinny projection kernel per compute unit
  int64_t w8a16_wide = 1;        // int8 codes read 16 per lane: 0 never, 1 for large matrices, 2 whenever shapes allow
  int64_t skinny_fuse = 7;         // skinny projections of up to four rows make their activations themselves: 1 norm, 2 SwiGLU, 4 merge
  int64_t skinny_fused = 0;        // read only: the sources that the last layer or FFN block took (bits as in skinny_fuse)
  int64_t w8a16_min_steps = 2;   // fewest 32-row steps per wavefront before k is split further
  int64_t gemm_stream = 1;         // projections of 33 to 96 rows that stream their weights: 0 never, 1 where measured ahead, 2 whenever shapes allow
  int64_t attn_order = -1;         // sequences by length: -1 where measured faster, 0 never, 1 always (partition grid and workgroup form)
  int64_t w8a16_gemm_rows = 33;  // rows from which int8 projections run as a tiled GEMM (0 = never)
};

Context& ctx();
// Host-side state (the scratch areas and their growth, the options, launch attributes set on first
// use) is shared by every caller, and a program's launches use the shared scratch areas in stream
// order.  Every entry point that sizes scratch or launches holds this lock for the duration of the
// call, so host threads take turns; it is recursive because pto_hip_run dispatches to the typed
// entry points.  The lock orders host work only: two streams still share one scratch area.
std::recursive_mutex& dispatch_mutex();
#define PTO_DISPATCH_LOCK() std::lock_guard<std::recursive_mutex> pto_dispatch_lock_(::pto_hip::dispatch_mutex())
// Returns a workspace of at least `bytes`.  A request beyond the current size allocates a new
// buffer of at least twice the old size and retires the old one without freeing it, so that
// queued work and launches recorded into a HIP graph stay valid; it fails while a stream is
// being captured (allocation is not allowed then): make each call once before capturing it.
int workspace(size_t bytes, void** ptr);

// ---- W8A16 decode projections, shared with the composed decoder layer -------------------
constexpr int kW8MaxM = 32;   // activation rows of the skinny kernels are at most this many
// Which workgroups of the skinny projection kernel share an output slab.  The (slab, 32-row k step) units of a
// launch form one list, slab by slab, and workgroup w of `wgs` takes the units [w * units / wgs,
// (w + 1) * units / wgs): a slab (2^shift channels, ks units) is the work of as many consecutive workgroups as
// its units fall to, and the j-th of them writes partial slab j.  units 0: every channel has `splits` slabs.
struct SlabMap {
  unsigned units, wgs, ks;
  int shift, slabs;  // slabs of one matrix (those of a pair's second matrix follow)
};
// Partial slabs of channel `ch` of matrix `mat`.
__device__ __forceinline__ int slab_count(const SlabMap& s, int splits, int mat, int ch) {
  if (s.units == 0) return splits;
  const unsigned first = (unsigned)(mat * s.slabs + (ch >> s.shift)) * s.ks;
  return (int)(((first + s.ks) * s.wgs - 1) / s.units - ((first + 1) * s.wgs - 1) / s.units) + 1;
}
// fp32 partial sums of a projection: element (s, m, n) of projection i is part[i][s * slab_stride + m * N + n] for
// s below slab_count(map, splits, i, n).  The skinny kernels write [M, N] slabs into the shared workspace; the
// tiled GEMM writes [M, N] slabs into its own scratch area (or, with one split, the finished product into the
// caller's buffer: `scaled` then says the channel scales are in).
struct W8Partials {
  float* part[2];
  int splits;
  int64_t slab_stride;
  bool scaled;
  SlabMap map;
};
// A finished fp32 product as a single slab.
inline W8Partials finished_slab(const float* product) {
  W8Partials p{};
  p.part[0] = const_cast<float*>(product);
  p.splits = 1;
  return p;
}
// Unmerged partials of an attention launch: per (sequence, query head) and partition the running maximum and sum, and the
// unnormalised result; partition i of a sequence holds tokens [i tpp, (i + 1) tpp) of its first ctx_cap.
struct AttnPartials {
  const float* ml;  // [B * Hq, n_part, 2]
  const float* o;   // [B * Hq, n_part, D]
  const int32_t* ctx_lens;
  int n_part, tpp, ctx_cap;
};
// What the workgroups of a skinny projection of up to kSkinnyFusedRows rows make their activations from (skinny.h).
constexpr int kSkinnyFusedRows = 4;
struct ProjectionSource {
  enum Kind { kTensor, kNorm, kSwiglu, kMerge } kind;
  const float* gamma;  // kNorm: x is the row-major input of the norm
  float eps;
  W8Partials pair;  // kSwiglu: the gate/up pair's partial slabs and scales
  const float* scale0;
  const float* scale1;
  AttnPartials attn;  // kMerge
  int head_dim;
};
// Whether a projection [m, k] @ [k, n] may be given the source (head_dim: kMerge only).
bool skinny_fuses(ProjectionSource::Kind kind, int64_t m, int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16, int64_t head_dim = 0);
constexpr int kMergeHeld = 40;  // most partitions per row of a kMerge source
// Bytes of the partial slabs of such a projection (up to kSkinnyFusedRows rows), for callers that provide the area: what a source is
// read from lies in workspace() itself.
size_t skinny_fused_bytes(int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16);
// Launches the partial kernel for x[M, K] @ wq0[K, N] (and wq1 when non-null).  x_blocked: x is
// stored [K/8][32][8] - element (m, k) at ((k/8)*32 + m)*8 + k%8 - the layout the layer's own
// producers write so that a wavefront's activation reads are whole consecutive cache lines.
// w16: the weights are 16-bit values of the activation type instead of int8 codes (the finish
// kernels then take null scales).
// src: the activations are made by the workgroups (x unused but for kNorm); area: where the slabs go instead of workspace().
int w8a16_partials(const void* x, bool x_blocked, const void* wq0, const void* wq1, int64_t m, int64_t k,
                   int64_t n, int x_dtype, hipStream_t st, W8Partials* out, bool w16 = false,
                   const ProjectionSource* src = nullptr, float* area = nullptr);
// Whether `st` is being captured (or that cannot be told).
bool stream_capturing(hipStream_t st);
// Grow-only device scratch for intermediates that must survive calls which use workspace().
int layer_workspace(size_t bytes, void** ptr);
// Grow-only device scratch for the split-K slabs of the tiled GEMMs.  Null when `st` is being captured and the area
// would have to grow: the product then runs unsplit.
int gemm_slabs(size_t bytes, hipStream_t st, void** ptr);
// out_rows of these and of the kernels below: 0 writes rows, otherwise the blocked layout [N/8][out_rows][8] of the next projection.
// out = cast(sum_s(part0) * scale0 [-> SiLU(.) * (sum_s(part1) * scale1)] [+ residual]).
int w8a16_finish(const W8Partials& parts, const float* scale0, const float* scale1, const void* residual,
                 int res_dtype, void* out, int out_dtype, int out_rows, int64_t m, int64_t n, hipStream_t st);
// sum_out = sum_s(part) * scale + residual (fp32); normed_out = cast(RMSNorm(sum_out) * gamma).
bool w8a16_finish_norm_fits(int64_t n);
int w8a16_finish_norm(const W8Partials& parts, const float* scale, const void* residual, int res_dtype,
                      float* sum_out, const float* gamma, void* normed_out, int out_dtype, int out_rows,
                      int64_t m, int64_t n, float eps, hipStream_t st);
// The tiled GEMM with int8 weight codes (widened on their way into LDS, scales applied to the
// accumulators): out = (x @ codes0) * scale0 (+ residual), or with codes1 / scale1 given
// SiLU((x @ codes0) * scale0) * ((x @ codes1) * scale1).  gemm_w8_fits says whether the shapes,
// types and addresses allow it; callers fall back to 32-row passes otherwise.
bool gemm_w8_fits(const void* x, const void* wq0, const void* wq1, const void* residual, const void* out, int64_t m,
                  int64_t k, int64_t n, int x_dtype, int out_dtype);
int gemm_w8(const void* x, const void* wq0, const float* scale0, const void* wq1, const float* scale1,
            const void* residual, int res_dtype, void* out, int64_t m, int64_t k, int64_t n, int x_dtype,
            int out_dtype, hipStream_t st);
// Projections of some tens of rows bound by reading their weights (stream_rows.h), left as fp32 slabs of k splits.  stream_rows_for
// says whether one is to run so - row count of the blocked layout its activations should have, 0 otherwise - and has made room
// for its slabs; x_rows: 0 for activations in rows.
int stream_rows_for(int64_t m, int64_t k, int64_t n, const void* wq0, const void* wq1, bool w16, hipStream_t st);
int stream_partials(const void* x, int x_rows, const void* wq0, const void* wq1, int64_t m, int64_t k, int64_t n, int x_dtype,
                    hipStream_t st, W8Partials* out, bool w16);
// x[M, K] @ w[K, N] through the tiled GEMM, left as k-split partial sums for a fused consumer
// (scale null: 16-bit weights).  With one split the product, scales applied, is written to
// `direct` (fp32 [M, N]) and returned as a single slab.
int gemm_partials(const void* x, const void* w, const float* scale, int64_t m, int64_t k, int64_t n, int x_dtype,
                  float* direct, hipStream_t st, W8Partials* out);

// RoPE + K/V append reading either final fp32 projections (qkv_scale null, splits 1) or the
// partial sums of the q/k/v projection (summed in split order and scaled per channel).
// rope_width: columns of the cos/sin tables, head_dim / 2 or head_dim.
int rope_kv_cache_update(const W8Partials& qkv, const float* qkv_scale,
                         const int32_t* seq_lens, const float* rope_cos, const float* rope_sin,
                         const int32_t* block_table, void* key_cache, void* value_cache, void* q_out,
                         int64_t batch, int64_t num_heads, int64_t kv_head_num, int64_t head_dim,
                         int64_t block_size, int64_t max_num_blocks_per_req, int64_t max_pos, int rope_width,
                         int64_t pool_rows, int dtype, void* stream);
int rope_kv_cache_update_fp8(const W8Partials& qkv, const float* qkv_scale,
                             const int32_t* seq_lens, const float* rope_cos, const float* rope_sin,
                             const int32_t* block_table, void* key_cache, void* value_cache, float* k_scale,
                             float* v_scale, void* q_out, int64_t batch, int64_t num_heads, int64_t kv_head_num,
                             int64_t head_dim, int64_t block_size, int64_t max_num_blocks_per_req,
                             int64_t max_pos, int rope_width, int64_t pool_blocks, int q_dtype, void* stream);
// RMSNorm of at most out_rows rows written in the blocked activation layout [H/8][out_rows][8].
bool rms_norm_blocked_fits(int64_t rows, int64_t hidden, int out_rows = kW8MaxM);
int rms_norm_blocked(const void* x, const float* gamma, void* out, int64_t rows, int64_t hidden, float eps,
                     int dtype, hipStream_t st, int out_rows = kW8MaxM);
// Rows of 16-bit values in that layout, as they are (hidden % 8 == 0, 16-byte aligned).
int rows_blocked(const void* x, void* out, int64_t rows, int64_t hidden, hipStream_t st, int out_rows);
int cast_from_f32(const float* in, void* out, size_t n, int out_dtype, hipStream_t st);
// pto_hip_paged_attention with an optional second output: the result rounded to the query dtype.
// out16_rows asks for the copy as [Hq*D/8][out16_rows][8] over the batch rows (at most so many);
// *wrote_blocked says whether that is how it was written (only a launch with a merge kernel can).
// pool_blocks > 0: the number of physical blocks in the caches; a table entry beyond it that a
// sequence uses reads block 0 instead and is reported by the next pto_hip_sync.
// active_blocks >= 0: no sequence attends beyond its first active_blocks blocks (the bound the SPMD
// form of the orchestration carries in its config, 09_paged_attention_spmd.py:468,482); < 0: no bound.
int paged_attention(const void* query, const void* key_cache, const void* value_cache,
                    const int32_t* block_table, const int32_t* context_lens, float* out, void* out16,
                    int out16_rows, bool* wrote_blocked,
                    const int64_t* config, int q_dtype, int kv_dtype, const float* k_scale,
                    const float* v_scale, int64_t pool_blocks, void* stream, void* fixed_scratch = nullptr,
                    size_t fixed_scratch_bytes = 0, int64_t active_blocks = -1, AttnPartials* unmerged = nullptr);
// unmerged: the caller can take the partials as they are, up to unmerged->n_part per row.  A launch that has a merge kernel and is
// not being measured then leaves it out and describes them there, `out` and `out16` unwritten; otherwise n_part comes back 0.
// Forgets every measured launch shape (and releases the events of measurements in flight).
void attention_tuning_reset();
// Residency cap, form (1 = workgroup form) and order (1 = sequences by length) the last launch's signature was tuned to; -1 while untuned.
void attention_tuning_last(int64_t* cap, int64_t* wg, int64_t* ordered);
// The same contract for the shapes the tiled kernels are not built for (head_dim other than 128 / 256
// up to 256, block sizes off the 16-token grid); attention_needs_generic says which launches take it.
bool attention_needs_generic(const int64_t* config, int kv_dtype);
int paged_attention_generic(const void* query, const void* key_cache, const void* value_cache,
                            const int32_t* block_table, const int32_t* context_lens, float* out,
                            const int64_t* config, int q_dtype, int kv_dtype, const float* k_scale,
                            const float* v_scale, int64_t pool_blocks, int64_t active_blocks, hipStream_t stream);
// fixed_scratch != null: the partition partials go there instead of the grow-only workspace, and a
// launch that needs more than fixed_scratch_bytes is refused (nothing is allocated either way).
//
// Looks up, for `device` (which must be current), the address of the file-scope device array that
// backs pto_hip_paged_attention_noalloc.  Called by pto_hip_init; idempotent per device.
int attn_static_scratch_init(int device);

inline int dtype_bytes(int dt) {
  switch (dt) {
    case PTO_HIP_INT8:
    case PTO_HIP_FP8E4M3FN:
      return 1;
    case PTO_HIP_FP16:
    case PTO_HIP_BF16:
      return 2;
    case PTO_HIP_INT32:
    case PTO_HIP_FP32:
      return 4;
    case PTO_HIP_INT64:
      return 8;
    default:
      return 0;
  }
}

inline const char* dtype_name(int dt) {
  switch (dt) {
    case PTO_HIP_INT8: return "INT8";
    case PTO_HIP_INT32: return "INT32";
    case PTO_HIP_INT64: return "INT64";
    case PTO_HIP_FP8E4M3FN: return "FP8E4M3FN";
    case PTO_HIP_FP16: return "FP16";
    case PTO_HIP_FP32: return "FP32";
    case PTO_HIP_BF16: return "BF16";
    default: return "?";
  }
}

}  // namespace pto_hip

// FFN block on e4m3 operands (no counterpart in the reference, whose FFN is 16-bit: this is the
// "fp8 MFMA" form of examples/models/01_ffn.py:111-131 / qwen3_jit/kernels/mlp.py:22-61).
//
//   xn  = bf16(RMSNorm(x) * gamma)                 one row kernel, which also quantises:
//   x8  = e4m3(xn / sx),  sx[t] = amax_row(xn) / 448
//   g,u = (x8 @ Wg8^T) * sx[t] * sg[n],  (x8 @ Wu8^T) * sx[t] * su[n]      fp32 accumulation
//   h   = bf16(SiLU(g) * u)                        epilogue of the gate/up GEMM
//   h8  = e4m3(h / sh),   sh[t] = amax_row(h) / 448                        row kernel
//   out = (h8 @ Wd8^T) * sh[t] * sd[n]
//
// Weights are e4m3 codes stored one row per OUTPUT channel with k contiguous ([out, in], i.e. the
// transpose of the 16-bit layout) plus one fp32 scale per output channel, so both GEMM operands
// are k-major and go global -> LDS -> registers without any transpose.  The GEMM uses
// v_mfma_f32_32x32x64_f8f6f4: lane l holds row/column l % 32 and the 32 codes k = 32 * (l / 32) .. +32.
// Products of a small call go to narrow_gemm8.h instead (choose_narrow8).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.h"
#include "launch_choice.h"
#include "lds_load.h"

namespace pto_hip {
namespace gemm8 {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef __attribute__((address_space(3))) const char lds_cchar;
typedef __attribute__((address_space(3))) const u32x4 lds_cu32x4;

constexpr int BK = 128;   // k extent of one LDS tile row, in codes (= bytes)
constexpr int BN = 256;   // B rows (output channels) per tile
constexpr int kXcds = 8;
constexpr float kE4m3Max = 448.f;

struct Params {
  const uint8_t* a;    // [M, K] codes, k contiguous
  const uint8_t* b0;   // [N, K] codes, one row per output channel
  const uint8_t* b1;   // gate/up pass: the up weights
  const float* sa;     // [M] row scales of a
  const float* sb0;    // [N] channel scales of b0
  const float* sb1;
  void* c;             // [M, N]
  int64_t lda, ldb, ldc;
  int m, n, k;
  int tiles_m, tiles_n;
  // k split over `splits` workgroups per output tile: each writes its raw fp32 accumulators to its own slab
  // ([split][m][n]; in the gate/up pass [split][2][m][n], gate then up); a finish kernel sums the slabs in
  // split order and applies the scales.  splits == 1: the epilogue finishes the tile.
  int splits, k_per_split;
  float* slabs;
};

// SiLU in the device form of the reference, g * recip(1 + exp(-g)) (01_ffn.py:70-74), with the hardware's
// 1-ulp reciprocal: the correctly rounded one is a ten-instruction division, and an epilogue computes
// 64 of them per lane while the matrix pipes idle.
__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

// two outputs rounded to the 16-bit type, packed
template <typename OutT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (OutT)a) | ((uint32_t)__builtin_bit_cast(uint16_t, (OutT)b) << 16);
}

// four consecutive outputs of one row as one store
template <typename OutT>
__device__ __forceinline__ void store4(OutT* dst, const float (&v)[4]) {
  if constexpr (sizeof(OutT) == 4) {
    *reinterpret_cast<float4*>(dst) = float4{v[0], v[1], v[2], v[3]};
  } else {
    const uint2 w = {pack2<OutT>(v[0], v[1]), pack2<OutT>(v[2], v[3])};
    *reinterpret_cast<uint2*>(dst) = w;
  }
}

__device__ __forceinline__ int xcd_remap(int pid, int nwg) {
  const int x = pid % kXcds, local = pid / kXcds;
  const int full = nwg / kXcds, rem = nwg % kXcds;
  const int base = x < rem ? x * (full + 1) : rem * (full + 1) + (x - rem) * full;
  return base + local;
}

template <int N>
struct Const {
  static constexpr int value = N;
};

// Tile (128*MH) x 256 x 128 on four wavefronts, one per SIMD, in a 2 x 2 grid; a wavefront owns
// (64*MH) x 128 as four quadrants of MH x 2 accumulators (32 x 32 each).  Row and column halves of a
// tile are the unit of everything: the operand tiles are cut into quarters A0, A1 (64*MH rows) and
// B0, B1 (128 channels) of whole 128-byte rows, and a k-tile is four phases
//     P1 (A0,B0)   P2 (A0,B1)   P3 (A1,B1)   P4 (A1,B0)
// of 4*MH MFMAs per wavefront.  The fragments of one quarter are read from LDS in the phase before
// their first use (P1 reads B1, P2 A1, P3 the next tile's A0, P4 its B0), so after each phase's barrier
// one quarter's slot is free and is requested again at once, RING tiles ahead: a request has
// 4*RING - 1 phases to land, and the waits (vmcnt counted, never 0) leave all but the oldest quarter
// in flight.  What bounds it: with whole tiles double-buffered instead (eight wavefronts of 128 x 64, one
// barrier and one full wait a k-tile), a k-tile took the 1.3-1.4 us that its 64 KB need to arrive,
// whatever its height, against 0.86 us of MFMA at the full clock; now the matrix pipes are busy in 77 % of
// the clocks of the gate/up pass and 74 % of the down pass's (SQ_VALU_MFMA_BUSY_CYCLES / 4 / SQ_BUSY_CU_CYCLES), and
// the shader clock drops to 2.0 GHz under the load.
// Weights of three blocks in turn, LLaMA-7B shape at 2048 tokens: gate/up pass 171 -> 148 us (2.5 PFLOP/s), down
// pass 119 -> 92 us, block 313 -> 264 us; at 300 / 512 / 1024 / 4000 tokens 129 -> 107, 148 -> 125, 193 -> 174,
// 527 -> 491 us.  Holding a whole tile's fragments (A0, A1, B0, B1) takes 96-128 registers next to 256
// accumulators: hence one wavefront per SIMD, which also reads a third less from LDS per MFMA than
// two of 128 x 64 would.
// The weights are the MFMA's first operand, so that an accumulator register holds four consecutive channels of
// one row: rows are stored 16 bytes at a time without a transpose (the matrix pipes wait out a tile's epilogue).
// In the gate/up pass a B quarter is 64 gate channels followed by the 64 up channels of the same
// outputs, and the two accumulator columns of a quadrant are gate / up of the same 32 outputs, so
// SiLU(g) * u is applied on the accumulators.
// The tiles go global -> LDS directly (1 KB per wavefront instruction = 8 rows); the hardware fixes
// where a lane's 16 bytes land, so instead of padding, the lane whose bytes land in slot s of row r
// fetches logical chunk s ^ ((r / 2) % 8) and the fragment reads apply the same XOR: the 16 lanes the
// LDS checks together for bank conflicts (16 consecutive rows, one logical chunk, 256 bytes = all 64
// banks) then hit 16 different slots of 8 row pairs.
// LONG: rows so long that a tile's last one starts 2^32 bytes or more after its first (kLongRow): an address per lane
// and request instead of 32-bit offsets from the tile's base (for all shapes: LLaMA-7B block at 2048 tokens 266.9 -> 269.1
// us, 1024 x 2816 at 1024 tokens 38.3 -> 38.7).
template <int MH, int RING, bool DUAL, bool SPLIT, bool LONG, typename OutT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm8_kernel(Params p) {
  constexpr int BM = 128 * MH;
  constexpr int QA = 64 * MH * BK, QB = 128 * BK;  // bytes of an A and of a B quarter
  constexpr int TILE = 2 * (QA + QB);
  constexpr int NA = 2 * MH, NB = 4;               // requests of one wavefront for an A and for a B quarter
  extern __shared__ __attribute__((aligned(16))) uint8_t smem8[];  // [RING][A0 | A1 | B0 | B1], then the row and channel scales
  lds_cchar* lds0 = (lds_cchar*)smem8;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int ntiles = p.tiles_m * p.tiles_n;
  const int logical = xcd_remap(blockIdx.x, ntiles * p.splits);
  const int split = logical / ntiles, tile_id = logical % ntiles;
  // bands of eight row tiles, rows first: an XCD's 32 consecutive ids are 8 row tiles x 4 column tiles
  // whatever the height of the problem (walking whole columns would pull all of A through its L2 per column tile)
  const int per_band = 8 * p.tiles_n;
  const int band = tile_id / per_band, idx = tile_id - band * per_band;
  const int band_rows = min(8, p.tiles_m - band * 8);
  const int tn = idx / band_rows, tm = band * 8 + (idx - tn * band_rows);
  const int k_begin = split * p.k_per_split;  // this workgroup's k range: [k_begin, k_begin + nk * BK)
  const int nk = (min(p.k, k_begin + p.k_per_split) - k_begin) / BK;
  const int m0 = tm * BM;
  const int n0 = tn * (DUAL ? BN / 2 : BN);

  // The tile's row and channel scales go to LDS now (clamped past the end): fetched after the loop they
  // would cost two memory round trips with the matrix pipes idle.
  float* s_rows = reinterpret_cast<float*>(smem8 + RING * TILE);  // [BM]
  float* s_cols = s_rows + BM;                                    // [256], in the order of the tile's B rows
  for (int r = tid; r < BM; r += 256) s_rows[r] = p.sa[min(m0 + r, p.m - 1)];
  {
    const int h = tid >> 7, r = tid & 127;
    const int ch = min(n0 + (DUAL ? h * 64 + (r & 63) : tid), p.n - 1);
    s_cols[tid] = (DUAL && r >= 64 ? p.sb1 : p.sb0)[ch];
  }

  // ---- requests: instruction e of a quarter brings its rows 32 e + 8 wave + lane / 8; rows and channels
  // past the end are clamped (their products are not stored) ----
  const int q_row = wave * 8 + (lane >> 3);
  const int chunk = (lane & 7) ^ ((q_row >> 1) & 7);  // logical chunk whose slot this lane fills
  const uint8_t* base_a = p.a + (int64_t)m0 * p.lda + k_begin;
  const uint8_t* base_b0 = p.b0 + (int64_t)n0 * p.ldb + k_begin;
  const uint8_t* base_b1 = DUAL ? p.b1 + (int64_t)n0 * p.ldb + k_begin : base_b0;
  typedef typename std::conditional<LONG, int64_t, uint32_t>::type Offset;
  Offset va[2][NA], vb[2][NB];  // byte offsets from the tile's first row / channel
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int e = 0; e < NA; ++e)
      va[h][e] = (Offset)min(h * 64 * MH + e * 32 + q_row, p.m - 1 - m0) * (Offset)p.lda + chunk * 16;
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int r = e * 32 + q_row;
      vb[h][e] = (Offset)min(DUAL ? h * 64 + (r & 63) : h * 128 + r, p.n - 1 - n0) * (Offset)p.ldb + chunk * 16;
    }
  }
  const uint32_t lds_w = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds0 + wave * 1024);
  auto bring = [&](auto off_c, Offset off, const uint8_t* base) {
    constexpr int OFF = decltype(off_c)::value;
    if constexpr (LONG) to_lds<OFF>(base + off, lds_w);
    else to_lds<OFF>(off, base, lds_w);
  };
  // request e of quarter Q (0 A0, 1 B0, 2 B1, 3 A1) of tile t (past the last one: the last again) into ring slot S
  auto request = [&](auto s_c, auto q_c, auto e_c, int t) {
    constexpr int S = decltype(s_c)::value, Q = decltype(q_c)::value, E = decltype(e_c)::value;
    const int koff = min(t, nk - 1) * BK;
    if constexpr (Q == 0 || Q == 3) {
      if constexpr (E < NA) bring(Const<S * TILE + (Q ? QA : 0) + E * 4096>{}, va[Q ? 1 : 0][E], base_a + koff);
    } else {
      bring(Const<S * TILE + 2 * QA + (Q - 1) * QB + E * 4096>{}, vb[Q - 1][E], (DUAL && E >= 2 ? base_b1 : base_b0) + koff);
    }
  };
  auto request_all = [&](auto s_c, auto q_c, int t) {
    request(s_c, q_c, Const<0>{}, t);
    request(s_c, q_c, Const<1>{}, t);
    request(s_c, q_c, Const<2>{}, t);
    request(s_c, q_c, Const<3>{}, t);
  };

  // ---- fragments: lane l holds row / channel l % 32, logical chunks 4 ks + 2 (l / 32) and the next; every
  // fragment starts at a row that is a multiple of 32, so the swizzle key is (l / 2) % 8 for all of them.
  // An LDS instruction reaches 64 KB past its address register: one register per 64 KB. ----
  constexpr int kReach = (RING * TILE + 65535) / 65536;
  lds_cchar* fa_base[kReach][4];
  lds_cchar* fb_base[kReach][4];
  {
    const int key = (lane >> 1) & 7;
#pragma unroll
    for (int w = 0; w < kReach; ++w)
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        const int c = 4 * (cc >> 1) + 2 * (lane >> 5) + (cc & 1);
        const int off = (lane & 31) * BK + ((c ^ key) << 4) + w * 65536;
        fa_base[w][cc] = lds0 + wm * (32 * MH) * BK + off;
        fb_base[w][cc] = lds0 + wn * (DUAL ? 32 : 64) * BK + off;
      }
  }
  v8i fa[2][MH][2], fb[2][2][2];  // [half or register set][fragment][k-step]
  // one 16-byte read: number i of quarter Q's 8 (A: 4 MH), into register set `set`
  auto read_one = [&](auto s_c, auto q_c, auto set_c, auto i_c) {
    constexpr int S = decltype(s_c)::value, Q = decltype(q_c)::value, SET = decltype(set_c)::value, I = decltype(i_c)::value;
    constexpr int F = I >> 2, CC = I & 3;
    if constexpr (Q == 0 || Q == 3) {
      if constexpr (F < MH) {
        constexpr int OFF = S * TILE + (Q ? QA : 0) + F * 32 * BK;
        const u32x4 v = *reinterpret_cast<lds_cu32x4*>(fa_base[OFF >> 16][CC] + (OFF & 65535));
#pragma unroll
        for (int w = 0; w < 4; ++w) fa[SET][F][CC >> 1][(CC & 1) * 4 + w] = (int)v[w];
      }
    } else {
      constexpr int OFF = S * TILE + 2 * QA + (Q - 1) * QB + F * (DUAL ? 64 : 32) * BK;
      const u32x4 v = *reinterpret_cast<lds_cu32x4*>(fb_base[OFF >> 16][CC] + (OFF & 65535));
#pragma unroll
      for (int w = 0; w < 4; ++w) fb[SET][F][CC >> 1][(CC & 1) * 4 + w] = (int)v[w];
    }
  };
  auto read_all = [&](auto s_c, auto q_c, auto set_c) {
    read_one(s_c, q_c, set_c, Const<0>{});
    read_one(s_c, q_c, set_c, Const<1>{});
    read_one(s_c, q_c, set_c, Const<2>{});
    read_one(s_c, q_c, set_c, Const<3>{});
    read_one(s_c, q_c, set_c, Const<4>{});
    read_one(s_c, q_c, set_c, Const<5>{});
    read_one(s_c, q_c, set_c, Const<6>{});
    read_one(s_c, q_c, set_c, Const<7>{});
  };

  f32x16 acc[2][MH][2][2];  // [row half][row fragment][column half][column fragment]
#pragma unroll
  for (int i = 0; i < 8 * MH; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) (&acc[0][0][0][0])[i][r] = 0.f;

  // Quarters in the order they are requested and read: u = 4 t + {0 A0, 1 B0, 2 B1, 3 A1} of tile t.
  // Requests of the n quarters after quarter u:
  constexpr auto in_flight = [](int u, int n) {
    int c = 0;
    for (int i = 1; i <= n; ++i) c += ((u + i) % 4 == 0 || (u + i) % 4 == 3) ? NA : NB;
    return c;
  };
  // One phase: quadrant (HA, HB) of the tile whose B halves sit in register sets PAR (B0) and 1 - PAR (B1);
  // reads quarter RQ from ring slot RS into register set RSET; requests quarter GQ of tile gt into slot GS.
  auto phase = [&](auto ha_c, auto hb_c, auto bset_c, auto rs_c, auto rq_c, auto rset_c, auto gs_c, auto gq_c, int gt) {
    constexpr int HA = decltype(ha_c)::value, HB = decltype(hb_c)::value, BS = decltype(bset_c)::value;
    auto slot = [&](auto q_c) {
      constexpr int q = decltype(q_c)::value;
      constexpr int ks = q / (2 * MH), i = (q % (2 * MH)) / 2, j = q % 2;
      acc[HA][i][HB][j] =
          __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[BS][j][ks], fa[HA][i][ks], acc[HA][i][HB][j], 0, 0, 0, 0, 0, 0);
      // the eight reads (four for a short A quarter) go with the first MFMAs, so that they have
      // landed when the phase ends; the requests one to an MFMA from the first
      if constexpr (q < 4) {
        read_one(rs_c, rq_c, rset_c, Const<2 * (q & 3)>{});
        read_one(rs_c, rq_c, rset_c, Const<2 * (q & 3) + 1>{});
        request(gs_c, gq_c, Const<(q & 3)>{}, gt);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    slot(Const<0>{});
    slot(Const<1>{});
    slot(Const<2>{});
    slot(Const<3>{});
    if constexpr (MH == 2) {
      slot(Const<4>{});
      slot(Const<5>{});
      slot(Const<6>{});
      slot(Const<7>{});
    }
    // the quarter the next phase reads has landed (this wavefront's part), this phase's reads are in registers
    constexpr int RQ = decltype(rq_c)::value;
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(in_flight(RQ + 1, 4 * RING - 2)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // Prologue: the first RING tiles requested, A0 and B0 of tile 0 read, A0 of tile RING requested.
  auto prologue = [&](auto s_c) {
    constexpr int S = decltype(s_c)::value;
    if constexpr (S < RING) {
      request_all(s_c, Const<0>{}, S);
      request_all(s_c, Const<1>{}, S);
      request_all(s_c, Const<2>{}, S);
      request_all(s_c, Const<3>{}, S);
    }
  };
  prologue(Const<0>{});
  prologue(Const<1>{});
  prologue(Const<2>{});
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(in_flight(2, 4 * RING - 3)) : "memory");  // quarters 0, 1, 2 have landed
  __builtin_amdgcn_sched_barrier(0);
  read_all(Const<0>{}, Const<0>{}, Const<0>{});
  read_all(Const<0>{}, Const<1>{}, Const<0>{});
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  request_all(Const<0>{}, Const<0>{}, RING);

  auto k_tile = [&](auto s_c, auto par_c, int t) {
    constexpr int S = decltype(s_c)::value, PAR = decltype(par_c)::value, S1 = (S + 1) % RING;
    typedef Const<0> C0;
    typedef Const<1> C1;
    //    quadrant        B regs            reads                                  requests
    phase(C0{}, C0{}, Const<PAR>{}, s_c, Const<2>{}, Const<1 - PAR>{}, s_c, Const<1>{}, t + RING);
    phase(C0{}, C1{}, Const<1 - PAR>{}, s_c, Const<3>{}, C1{}, s_c, Const<2>{}, t + RING);
    phase(C1{}, C1{}, Const<1 - PAR>{}, Const<S1>{}, Const<0>{}, C0{}, s_c, Const<3>{}, t + RING);
    phase(C1{}, C0{}, Const<PAR>{}, Const<S1>{}, Const<1>{}, Const<1 - PAR>{}, Const<S1>{}, Const<0>{}, t + 1 + RING);
  };
  if constexpr (RING == 2) {
    int t = 0;
    for (; t + 1 < nk; t += 2) {
      k_tile(Const<0>{}, Const<0>{}, t);
      k_tile(Const<1>{}, Const<1>{}, t + 1);
    }
    if (t < nk) k_tile(Const<0>{}, Const<0>{}, t);
  } else {
    int t = 0;
    for (; t + 5 < nk; t += 6) {
      k_tile(Const<0>{}, Const<0>{}, t);
      k_tile(Const<1>{}, Const<1>{}, t + 1);
      k_tile(Const<2>{}, Const<0>{}, t + 2);
      k_tile(Const<0>{}, Const<1>{}, t + 3);
      k_tile(Const<1>{}, Const<0>{}, t + 4);
      k_tile(Const<2>{}, Const<1>{}, t + 5);
    }
    if (t < nk) k_tile(Const<0>{}, Const<0>{}, t);
    if (t + 1 < nk) k_tile(Const<1>{}, Const<1>{}, t + 1);
    if (t + 2 < nk) k_tile(Const<2>{}, Const<0>{}, t + 2);
    if (t + 3 < nk) k_tile(Const<0>{}, Const<1>{}, t + 3);
    if (t + 4 < nk) k_tile(Const<1>{}, Const<0>{}, t + 4);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS after this
  __syncthreads();

  // ---- epilogue ----------------------------------------------------------------------------------
  // acc[ha][i][hb][j][r]: row m0 + ha*64*MH + wm*32*MH + i*32 + lane%32, channel (r/4)*8 + (lane/32)*4 + r%4 of its
  // fragment: a lane owns whole runs of four channels of one row.  The matrix pipes idle meanwhile, so a
  // lane's first address is computed once, every other one is a wave-uniform distance away, and only tiles at
  // the right and lower edge check bounds.
  constexpr int JN = DUAL ? 1 : 2;          // output fragments of a quadrant
  constexpr int HC = DUAL ? 64 : 128;       // output channels of a column half
  const int c_row = m0 + wm * 32 * MH + (lane & 31), c_col = n0 + wn * (DUAL ? 32 : 64);
  const int hi = lane >> 5;
  if constexpr (SPLIT) {
    // raw accumulators to this split's slab (n % 4 == 0)
    const int64_t mn = (int64_t)p.m * p.n;
    float* mine = p.slabs + (int64_t)split * (DUAL ? 2 : 1) * mn + (int64_t)c_row * p.n + c_col + hi * 4;
#pragma unroll
    for (int ha = 0; ha < 2; ++ha)
#pragma unroll
      for (int i = 0; i < MH; ++i) {
        float* dst = mine + (int64_t)(ha * 64 * MH + i * 32) * p.n;
        if (c_row + ha * 64 * MH + i * 32 >= p.m) continue;
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x16& t = acc[ha][i][hb][j];
              const int cc = hb * HC + (DUAL ? 0 : j * 32) + q * 8;
              if (c_col + hi * 4 + cc < p.n)
                *reinterpret_cast<float4*>(dst + (DUAL && j ? mn : 0) + cc) = float4{t[q * 4], t[q * 4 + 1], t[q * 4 + 2], t[q * 4 + 3]};
            }
      }
  } else {
    float sr[2][MH];  // this lane's row scales
#pragma unroll
    for (int ha = 0; ha < 2; ++ha)
#pragma unroll
      for (int i = 0; i < MH; ++i) sr[ha][i] = s_rows[wm * 32 * MH + ha * 64 * MH + i * 32 + (lane & 31)];
    OutT* c = reinterpret_cast<OutT*>(p.c);
    auto finish = [&](auto check_c) {
      constexpr bool CHECK = decltype(check_c)::value != 0;
      constexpr int VEC = 16 / (int)sizeof(OutT);  // elements of a lane's store
      const bool vec = !CHECK || (p.n % VEC == 0 && p.ldc % VEC == 0);
      OutT* lane_c = c + (int64_t)c_row * p.ldc + c_col + hi * VEC;
#pragma unroll
      for (int hb = 0; hb < 2; ++hb)
#pragma unroll
        for (int j = 0; j < JN; ++j) {
          const int cc0 = hb * HC + j * 32;
          float s0[16], s1[16];  // channel scales of this fragment (gate, up)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float* src = s_cols + hb * 128 + (DUAL ? wn * 32 : wn * 64 + j * 32) + q * 8 + hi * 4;
            *reinterpret_cast<float4*>(&s0[q * 4]) = *reinterpret_cast<const float4*>(src);
            if constexpr (DUAL) *reinterpret_cast<float4*>(&s1[q * 4]) = *reinterpret_cast<const float4*>(src + 64);
          }
#pragma unroll
          for (int ha = 0; ha < 2; ++ha)
#pragma unroll
            for (int i = 0; i < MH; ++i) {
              const int rr = ha * 64 * MH + i * 32;
              OutT* dst = lane_c + (int64_t)rr * p.ldc + cc0;
              float v[16];
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                if constexpr (DUAL) {
                  const float g = acc[ha][i][hb][0][r] * sr[ha][i] * s0[r], u = acc[ha][i][hb][1][r] * sr[ha][i] * s1[r];
                  v[r] = silu(g) * u;
                } else {
                  v[r] = acc[ha][i][hb][j][r] * sr[ha][i] * s0[r];
                }
              }
              if (vec) {
                if (CHECK && c_row + rr >= p.m) continue;
                if constexpr (sizeof(OutT) == 4) {
#pragma unroll
                  for (int q = 0; q < 4; ++q)
                    if (!CHECK || c_col + hi * 4 + cc0 + q * 8 < p.n)
                      *reinterpret_cast<float4*>(dst + q * 8) = float4{v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]};
                } else {
                  // the two halves of the wavefront trade runs, so that a lane stores eight channels at once
#pragma unroll
                  for (int q = 0; q < 4; q += 2) {
                    uint32_t w[2][2];
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                      const u32x2 x = __builtin_amdgcn_permlane32_swap(pack2<OutT>(v[q * 4 + 2 * d], v[q * 4 + 2 * d + 1]),
                                                                       pack2<OutT>(v[q * 4 + 4 + 2 * d], v[q * 4 + 5 + 2 * d]), false, false);
                      w[0][d] = x[0];
                      w[1][d] = x[1];
                    }
                    if (!CHECK || c_col + hi * 8 + cc0 + q * 8 < p.n)
                      *reinterpret_cast<u32x4*>(dst + q * 8) = u32x4{w[0][0], w[0][1], w[1][0], w[1][1]};
                  }
                }
              } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                  const int col = c_col + cc0 + (r >> 2) * 8 + hi * 4 + (r & 3);
                  if (c_row + rr < p.m && col < p.n) c[(int64_t)(c_row + rr) * p.ldc + col] = (OutT)v[r];
                }
              }
            }
        }
    };
    if (m0 + BM <= p.m && n0 + (DUAL ? BN / 2 : BN) <= p.n && p.ldc % (16 / (int)sizeof(OutT)) == 0) finish(Const<0>{});
    else finish(Const<1>{});
  }
}

constexpr int64_t kLongRow = (1ll << 32) / 256;  // rows of this many bytes and more: see LONG

template <int MH, bool DUAL, typename OutT, bool SPLIT = false, bool LONG = false>
int launch(Params p, hipStream_t st) {
  constexpr int BM = 128 * MH;
  constexpr int RING = MH == 2 ? 2 : 3;  // 128 or 144 KB of LDS
  p.tiles_m = (p.m + BM - 1) / BM;
  const int bn_out = DUAL ? BN / 2 : BN;
  p.tiles_n = (p.n + bn_out - 1) / bn_out;
  const size_t smem = (size_t)RING * (BM + BN) * BK + (BM + BN) * sizeof(float);
  auto kern = gemm8_kernel<MH, RING, DUAL, SPLIT, LONG, OutT>;
  static std::atomic<bool> attr_set{false};  // per instantiation; callers hold the dispatch lock
  if (!attr_set.load(std::memory_order_acquire)) {
    PTO_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)smem));
    attr_set.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3(p.tiles_m * p.tiles_n * p.splits), dim3(256), smem, st, p);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

// Four outputs of one row from the k splits' slabs: the sums in split order, times the row and channel
// scales (and SwiGLU for the gate/up pass, whose slabs are [split][2][m][n]).
template <bool DUAL>
__device__ __forceinline__ void sum_slabs(const float* src, int64_t mn, int splits, float row_scale, const float4& w0,
                                          const float4& w1, float (&out)[4]) {
  constexpr int kMats = DUAL ? 2 : 1;
  float4 t[kMats];
#pragma unroll
  for (int mat = 0; mat < kMats; ++mat) t[mat] = *reinterpret_cast<const float4*>(src + mat * mn);
  for (int s = 1; s < splits; ++s) {
#pragma unroll
    for (int mat = 0; mat < kMats; ++mat) {
      const float4 v = *reinterpret_cast<const float4*>(src + ((int64_t)s * kMats + mat) * mn);
      t[mat] = float4{t[mat].x + v.x, t[mat].y + v.y, t[mat].z + v.z, t[mat].w + v.w};
    }
  }
  const float r = row_scale;
  const float g[4] = {t[0].x * r * w0.x, t[0].y * r * w0.y, t[0].z * r * w0.z, t[0].w * r * w0.w};
  if constexpr (DUAL) {
    const float u[4] = {t[1].x * r * w1.x, t[1].y * r * w1.y, t[1].z * r * w1.z, t[1].w * r * w1.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = silu(g[k]) * u[k];
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = g[k];
  }
}

template <bool DUAL, typename OutT>
__global__ __launch_bounds__(256) void gemm8_finish_kernel(const float* __restrict__ slabs, int splits,
                                                           const float* __restrict__ sa, const float* __restrict__ sb0,
                                                           const float* __restrict__ sb1, OutT* __restrict__ c, int64_t ldc,
                                                           int m, int n) {
  // blockIdx.x, threadIdx.x: four columns; blockIdx.y: rows, strided (no division per element)
  const int col = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (col >= n) return;
  const int64_t mn = (int64_t)m * n;
  const float4 w0 = *reinterpret_cast<const float4*>(sb0 + col);
  const float4 w1 = DUAL ? *reinterpret_cast<const float4*>(sb1 + col) : w0;
  for (int64_t row = blockIdx.y; row < m; row += gridDim.y) {
    float out[4];
    sum_slabs<DUAL>(slabs + row * n + col, mn, splits, sa[row], w0, w1, out);
    store4<OutT>(c + row * ldc + col, out);
  }
}

}  // namespace gemm8
}  // namespace pto_hip

#include "narrow_gemm8.h"

namespace pto_hip {
namespace gemm8 {

// Picks the tile height and the k splits and launches the tiles.  With p.splits > 1 afterwards the slabs
// hold the raw sums and the caller finishes them: in a launch of its own, or (sums_on_the_way) in one that it makes anyway.
template <bool DUAL, typename OutT>
int launch_tiles(Params& p, bool sums_on_the_way, hipStream_t st) {
  const int64_t num_cu = pto_hip::ctx().num_cu, variant = pto_hip::ctx().gemm_variant, forced = pto_hip::ctx().gemm_splits;
  const int64_t tiles_n = (p.n + (DUAL ? 127 : 255)) / (DUAL ? 128 : 256);
  const int nk = p.k / BK;
  const bool can_split = p.n % 4 == 0 && p.ldc % 4 == 0;
  bool tall = variant != 5;
  int splits = can_split && nk >= 2 ? (int)std::min<int64_t>(std::max<int64_t>(forced, 1), nk) : 1;
  if (variant == 0) {
    // The pair of tile height and k splits with the least estimated time in microseconds: rounds of
    // workgroups over the CUs x (k-tiles x the time of one, growing with the share of CUs that are busy, plus a
    // tile's start and epilogue), not less than the weights take to arrive; with k split, plus the finish launch
    // and the slabs' way out and back.  Fitted at 8 to 4096 rows of four weight shapes (hidden
    // 1024 to 5120).  Timed against every pair at 8 to 4000 rows of five, the one it picks is 2.0 % from the best on
    // average and 21 % at worst in gate/up passes, 1.7 % and 17 % in single ones.
    const int from = forced > 0 ? splits : 1, to = forced > 0 ? splits : can_split ? std::max(1, std::min(16, nk / 2)) : 1;
    double best = 1e30;
    for (int th = 1; th >= 0; --th) {
      const int64_t tiles = (p.m + (th ? 255 : 127)) / (th ? 256 : 128) * tiles_n;
      for (int sp = from; sp <= to; ++sp) {
        const int64_t per = (nk + sp - 1) / sp, real = (nk + per - 1) / per, wgs = tiles * real;
        const double load = std::min(1.0, (double)wgs / (double)num_cu);
        const double tile_us = th ? 1.13 + 0.19 * load : 0.64 + 0.26 * load;
        double t = std::max((double)((wgs + num_cu - 1) / num_cu) * ((double)per * tile_us + (th ? 6.8 : 3.7)),
                            7.2 + (double)p.k * p.n * (DUAL ? 2 : 1) / 9.2e6);
        if (real > 1) t += 3.0 + 2.0 * (double)real * p.m * p.n * (DUAL ? 8 : 4) / 4.9e6;
        if (t < best) {
          best = t;
          tall = th != 0;
          splits = sp;
        }
      }
    }
    // Small calls in narrow tiles, one launch.  The estimate's 3 us for the launch that sums the slabs do not count against a caller that has one anyway.
    // (not a result laid over its own activations: one workgroup would write what another has still to read)
    const int64_t narrow = pto_hip::ctx().gemm_narrow;
    const uintptr_t a0 = (uintptr_t)p.a, c0 = (uintptr_t)p.c;
    const bool in_place = c0 < a0 + (uintptr_t)p.m * p.lda && a0 < c0 + (uintptr_t)p.m * p.ldc * sizeof(OutT);
    if (can_split && forced == 0 && narrow >= 0 && !in_place) {
      const double tiled_us = best - (sums_on_the_way && splits > 1 ? 3.0 : 0.0);
      const int tile = narrow > 0 ? (int)std::min<int64_t>(narrow, 3) : pto_hip::choose_narrow8(p.m, p.n, p.k, DUAL, num_cu, tiled_us);
      if (tile > 0) {
        p.splits = 1;
        return launch_narrow8<DUAL, OutT>(p, tile, st);
      }
    }
  }
  const bool long_rows = std::max(p.lda, p.ldb) >= kLongRow;  // built on 128-row tiles
  const int per = (nk + splits - 1) / splits;
  p.k_per_split = per * BK;
  p.splits = (nk + per - 1) / per;
  p.slabs = nullptr;
  if (p.splits > 1) {
    void* ws = nullptr;
    const int rc = pto_hip::gemm_slabs((size_t)p.splits * (DUAL ? 2 : 1) * p.m * p.n * sizeof(float), st, &ws);
    if (rc) return rc;
    p.slabs = reinterpret_cast<float*>(ws);
  }
  if (p.slabs) {
    if (long_rows) return launch<1, DUAL, float, true, true>(p, st);
    return tall ? launch<2, DUAL, float, true>(p, st) : launch<1, DUAL, float, true>(p, st);
  }
  p.splits = 1;
  p.k_per_split = p.k;
  if (long_rows) return launch<1, DUAL, OutT, false, true>(p, st);
  return tall ? launch<2, DUAL, OutT>(p, st) : launch<1, DUAL, OutT>(p, st);
}

template <bool DUAL, typename OutT>
int launch_any(Params p, hipStream_t st) {
  const int rc = launch_tiles<DUAL, OutT>(p, false, st);
  if (rc || p.splits == 1) return rc;
  const unsigned bx = (unsigned)((p.n / 4 + 255) / 256);
  const unsigned by = (unsigned)std::min<int64_t>(p.m, std::max<int64_t>(1, 4096 / bx));
  hipLaunchKernelGGL((gemm8_finish_kernel<DUAL, OutT>), dim3(bx, by), dim3(256), 0, st, p.slabs, p.splits, p.sa, p.sb0,
                     p.sb1, reinterpret_cast<OutT*>(p.c), p.ldc, p.m, p.n);
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

// ---- row kernels: (RMSNorm +) per-row e4m3 quantisation -----------------------------------------
constexpr int kRowThreads = 256;
constexpr int kRowVecs = 8;  // most 8-element groups a thread keeps in registers: rows of up to 16384 columns

__device__ __forceinline__ float clamp_e4m3(float v) { return fminf(fmaxf(v, -kE4m3Max), kE4m3Max); }

__device__ __forceinline__ float block_reduce(float v, bool take_max, float* shared) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float o = __shfl_xor(v, off);
    v = take_max ? fmaxf(v, o) : v + o;
  }
  if ((threadIdx.x & 63) == 0) shared[threadIdx.x >> 6] = v;
  __syncthreads();
  float tot = shared[0];
#pragma unroll
  for (int w = 1; w < kRowThreads / 64; ++w) tot = take_max ? fmaxf(tot, shared[w]) : tot + shared[w];
  return tot;
}

// One workgroup per row, the row held in registers.  NORM: y = T(x * rsqrt(mean x^2 + eps) * gamma)
// first (rounded to the 16-bit activation type, as the 16-bit block's RMSNorm output is); then
// scale = amax|y| / 448 (1 for an all-zero row) and codes = e4m3(clamp(y / scale)).
// SLABS: y = T(SwiGLU of the gate/up pass's k-split slabs), the row that gemm8_finish_kernel would write.
struct SlabRows {
  const float *slabs, *sa, *sb0, *sb1;  // [splits][2][rows][cols], row scales, channel scales of gate and up
  int64_t mn;                           // rows * cols
  int splits;
};
// VECS: groups of eight a thread holds, 2, 4 or 8.  The work on groups a row does not have and the registers they take are
// what bounded short rows.  Eight groups always -> now, bf16, with / without RMSNorm, us: 2048 x 4096 11.2 / 9.0 -> 9.2 / 8.0, 4000 x 2048 12.2
// / 10.1 -> 9.6 / 8.0, 4096 x 8192 28.6 / 21.1 -> 26.5 / 20.5; e4m3 FFN block of 2048 x 4096 x 11008 258.0 -> 256.6.  Six for rows of 8193 to 12288 columns
// loses: 2048 x 11008 24.0 / 16.5 -> 25.4 / 20.0.
template <typename TI, bool NORM, bool SLABS, int VECS>
__global__ __launch_bounds__(kRowThreads) void row_quant_kernel(const TI* __restrict__ x, const float* __restrict__ gamma,
                                                                uint8_t* __restrict__ codes, float* __restrict__ scale,
                                                                int64_t cols, float eps, SlabRows sl) {
  typedef __attribute__((__vector_size__(8 * sizeof(TI)))) TI vec8;
  __shared__ float red[2][kRowThreads / 64];
  const int64_t row = blockIdx.x;
  const vec8* xr = reinterpret_cast<const vec8*>(x + row * cols);
  const int nvec = (int)(cols / 8);
  // The row stays in registers in its 16-bit form (four registers per group of eight, not eight):
  // with the whole row's workgroups resident at once the kernel is one round of loads, not two.
  vec8 y[VECS];
  float ss = 0.f;
  constexpr bool kGammaAhead = NORM && VECS <= 4;  // requested with the row, as far as the registers for it go
  float4 ga[kGammaAhead ? 2 * VECS : 1];
  if constexpr (kGammaAhead) {
#pragma unroll
    for (int u = 0; u < VECS; ++u) {
      const int i = threadIdx.x + u * kRowThreads;
#pragma unroll
      for (int half = 0; half < 2; ++half)
        ga[2 * u + half] = gamma && i < nvec ? reinterpret_cast<const float4*>(gamma)[2 * i + half] : float4{1.f, 1.f, 1.f, 1.f};
    }
  }
#pragma unroll
  for (int u = 0; u < VECS; ++u) {
    const int i = threadIdx.x + u * kRowThreads;
    if (i < nvec) {
      if constexpr (SLABS) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int col = 8 * i + 4 * half;
          float v[4];
          sum_slabs<true>(sl.slabs + row * cols + col, sl.mn, sl.splits, sl.sa[row], *reinterpret_cast<const float4*>(sl.sb0 + col),
                          *reinterpret_cast<const float4*>(sl.sb1 + col), v);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[u][4 * half + e] = (TI)v[e];
        }
      } else {
        y[u] = xr[i];
      }
      if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)y[u][e] * (float)y[u][e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) y[u][e] = (TI)0.f;
    }
  }
  if constexpr (NORM) {
    const float inv = rsqrtf(block_reduce(ss, false, red[0]) / (float)cols + eps);
#pragma unroll
    for (int u = 0; u < VECS; ++u) {
      const int i = threadIdx.x + u * kRowThreads;
      if (i < nvec) {
        float4 g0, g1;
        if constexpr (kGammaAhead) {
          g0 = ga[2 * u];
          g1 = ga[2 * u + 1];
        } else {
          g0 = gamma ? reinterpret_cast<const float4*>(gamma)[2 * i] : float4{1.f, 1.f, 1.f, 1.f};
          g1 = gamma ? reinterpret_cast<const float4*>(gamma)[2 * i + 1] : float4{1.f, 1.f, 1.f, 1.f};
        }
        const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) y[u][e] = (TI)((float)y[u][e] * inv * g[e]);
      }
    }
  }
  float amax = 0.f;
#pragma unroll
  for (int u = 0; u < VECS; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf((float)y[u][e]));
  amax = block_reduce(amax, true, red[1]);
  const float s = amax > 0.f ? amax / kE4m3Max : 1.f;
  // y / s, correctly rounded, without the compiler's ten-instruction division per element: the
  // reciprocal of s is refined once per row to within half an ulp (one Newton step on v_rcp_f32), and
  // each quotient is q0 = y * r corrected twice by its exact remainder, q + (y - q * s) * r (two
  // fused multiply-adds each; one correction alone leaves a few quotients in ten million an ulp off).  |y| <= amax = 448 * s, so no quotient leaves [-448, 448]: nothing over- or
  // underflows, which is all the full sequence adds.
  float r = __builtin_amdgcn_rcpf(s);
  r = fmaf(fmaf(-s, r, 1.f), r, r);
  auto quot = [&](float v) {
    const float q0 = v * r;
    const float q1 = fmaf(fmaf(-q0, s, v), r, q0);  // within an ulp of v / s
    const float q2 = fmaf(fmaf(-q1, s, v), r, q1);  // its exact remainder settles the last bit
    return v == 0.f ? v : q2;                       // a zero keeps its sign (the corrections add +0 to -0)
  };
  if (threadIdx.x == 0) scale[row] = s;
  uint2* crow = reinterpret_cast<uint2*>(codes + row * cols);
#pragma unroll
  for (int u = 0; u < VECS; ++u) {
    const int i = threadIdx.x + u * kRowThreads;
    if (i < nvec) {
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = clamp_e4m3(quot((float)y[u][e]));
      int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
      w0 = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], w0, true);
      int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], 0, false);
      w1 = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], w1, true);
      crow[i] = uint2{(uint32_t)w0, (uint32_t)w1};
    }
  }
}

// Launches the instantiation for a row's length.
template <typename TI, bool NORM, bool SLABS>
void launch_row_quant(const void* x, const float* gamma, void* codes, float* scale, int64_t rows, int64_t cols, float eps,
                      const SlabRows& sl, hipStream_t st) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)rows), dim3(kRowThreads), 0, st, reinterpret_cast<const TI*>(x), gamma,
                       reinterpret_cast<uint8_t*>(codes), scale, cols, eps, sl);
  };
  const int64_t vecs = (cols / 8 + kRowThreads - 1) / kRowThreads;
  if (vecs <= 2) go(row_quant_kernel<TI, NORM, SLABS, 2>);
  else if (vecs <= 4) go(row_quant_kernel<TI, NORM, SLABS, 4>);
  else go(row_quant_kernel<TI, NORM, SLABS, kRowVecs>);
}

int row_quant(const void* x, const float* gamma, bool norm, void* codes, float* scale, int64_t rows, int64_t cols,
              float eps, int x_dtype, hipStream_t st) {
  PTO_CHECK_ARG(cols % 8 == 0 && cols <= 8 * kRowThreads * kRowVecs,
                "quantize_rows_fp8: %lld columns; rows must be a multiple of 8 and at most %d long", (long long)cols,
                8 * kRowThreads * kRowVecs);
  PTO_CHECK_ARG(rows < (1ll << 31), "quantize_rows_fp8: too many rows");
  PTO_CHECK_ARG(((uintptr_t)x | (uintptr_t)gamma) % 16 == 0 && (uintptr_t)codes % 8 == 0,
                "quantize_rows_fp8: misaligned operand");
  if (rows == 0) return PTO_HIP_OK;
  if (x_dtype == PTO_HIP_BF16) {
    if (norm) launch_row_quant<__bf16, true, false>(x, gamma, codes, scale, rows, cols, eps, SlabRows{}, st);
    else launch_row_quant<__bf16, false, false>(x, gamma, codes, scale, rows, cols, eps, SlabRows{}, st);
  } else if (x_dtype == PTO_HIP_FP16) {
    if (norm) launch_row_quant<_Float16, true, false>(x, gamma, codes, scale, rows, cols, eps, SlabRows{}, st);
    else launch_row_quant<_Float16, false, false>(x, gamma, codes, scale, rows, cols, eps, SlabRows{}, st);
  } else {
    return pto_hip::fail(PTO_HIP_ERR_INVALID_VALUE, "quantize_rows_fp8: dtype %s not in {BF16, FP16}",
                         pto_hip::dtype_name(x_dtype));
  }
  PTO_CHECK_HIP(hipGetLastError());
  return PTO_HIP_OK;
}

}  // namespace gemm8
}  // namespace pto_hip

extern "C" int pto_hip_quantize_rows_fp8(const void* x, void* codes, float* scale, int64_t rows, int64_t cols,
                                         int x_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  PTO_CHECK_ARG(rows >= 0 && cols > 0, "quantize_rows_fp8: bad shape [%lld, %lld]", (long long)rows, (long long)cols);
  if (rows == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(x && codes && scale, "quantize_rows_fp8: null tensor pointer");
  return gemm8::row_quant(x, nullptr, false, codes, scale, rows, cols, 0.f, x_dtype, (hipStream_t)stream);
}

extern "C" int pto_hip_rms_norm_quantize_fp8(const void* x, const float* gamma, void* codes, float* scale,
                                             int64_t rows, int64_t cols, float eps, int x_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  PTO_CHECK_ARG(rows >= 0 && cols > 0, "rms_norm_quantize_fp8: bad shape [%lld, %lld]", (long long)rows,
                (long long)cols);
  if (rows == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(x && codes && scale, "rms_norm_quantize_fp8: null tensor pointer");
  return gemm8::row_quant(x, gamma, true, codes, scale, rows, cols, eps, x_dtype, (hipStream_t)stream);
}

namespace {
int check_gemm8(const char* what, int64_t m, int64_t k, int64_t n, const void* a, const void* b, const void* c) {
  using namespace pto_hip;
  PTO_CHECK_ARG(m >= 0 && k > 0 && n > 0 && m < (1 << 30) && k < (1 << 30) && n < (1 << 30),
                "%s: bad shape M=%lld K=%lld N=%lld", what, (long long)m, (long long)k, (long long)n);
  if (k % gemm8::BK != 0)
    return fail(PTO_HIP_ERR_UNSUPPORTED, "%s: k %lld must be a multiple of %d", what, (long long)k, gemm8::BK);
  PTO_CHECK_ARG(((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) % 16 == 0, "%s: operand pointers must be 16-byte aligned",
                what);
  return PTO_HIP_OK;
}
}  // namespace

extern "C" int pto_hip_gate_up_swiglu_fp8(const void* x8, const float* x_scale, const void* w_gate8,
                                          const float* w_gate_scale, const void* w_up8, const float* w_up_scale,
                                          void* h, int64_t m, int64_t k, int64_t n, int h_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  int rc = check_gemm8("gate_up_swiglu_fp8", m, k, n, x8, w_gate8, h);
  if (rc) return rc;
  if (m == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(x8 && x_scale && w_gate8 && w_gate_scale && w_up8 && w_up_scale && h,
                "gate_up_swiglu_fp8: null tensor pointer");
  PTO_CHECK_ARG(((uintptr_t)w_up8 | (uintptr_t)w_gate_scale | (uintptr_t)w_up_scale) % 16 == 0,
                "gate_up_swiglu_fp8: operand and channel-scale pointers must be 16-byte aligned");
  PTO_CHECK_ARG(h_dtype == PTO_HIP_BF16 || h_dtype == PTO_HIP_FP16, "gate_up_swiglu_fp8: h dtype %s not in {BF16, FP16}",
                dtype_name(h_dtype));
  gemm8::Params p{};
  p.a = reinterpret_cast<const uint8_t*>(x8);
  p.b0 = reinterpret_cast<const uint8_t*>(w_gate8);
  p.b1 = reinterpret_cast<const uint8_t*>(w_up8);
  p.sa = x_scale;
  p.sb0 = w_gate_scale;
  p.sb1 = w_up_scale;
  p.c = h;
  p.lda = k;
  p.ldb = k;
  p.ldc = n;
  p.m = (int)m;
  p.n = (int)n;
  p.k = (int)k;
  hipStream_t st = (hipStream_t)stream;
  return h_dtype == PTO_HIP_BF16 ? gemm8::launch_any<true, __bf16>(p, st) : gemm8::launch_any<true, _Float16>(p, st);
}

extern "C" int pto_hip_projection_fp8(const void* a8, const float* a_scale, const void* w8, const float* w_scale,
                                      void* out, int64_t m, int64_t k, int64_t n, int out_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  int rc = check_gemm8("projection_fp8", m, k, n, a8, w8, out);
  if (rc) return rc;
  if (m == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(a8 && a_scale && w8 && w_scale && out, "projection_fp8: null tensor pointer");
  // the split-k finish and the tile epilogue read the channel scales four at a time
  PTO_CHECK_ARG((uintptr_t)w_scale % 16 == 0, "projection_fp8: the channel scales must be 16-byte aligned");
  gemm8::Params p{};
  p.a = reinterpret_cast<const uint8_t*>(a8);
  p.b0 = reinterpret_cast<const uint8_t*>(w8);
  p.sa = a_scale;
  p.sb0 = w_scale;
  p.c = out;
  p.lda = k;
  p.ldb = k;
  p.ldc = n;
  p.m = (int)m;
  p.n = (int)n;
  p.k = (int)k;
  hipStream_t st = (hipStream_t)stream;
  switch (out_dtype) {
    case PTO_HIP_FP32: return gemm8::launch_any<false, float>(p, st);
    case PTO_HIP_BF16: return gemm8::launch_any<false, __bf16>(p, st);
    case PTO_HIP_FP16: return gemm8::launch_any<false, _Float16>(p, st);
    default:
      return fail(PTO_HIP_ERR_INVALID_VALUE, "projection_fp8: output dtype %s not in {FP32, BF16, FP16}",
                  dtype_name(out_dtype));
  }
}

extern "C" int pto_hip_ffn_swiglu_fp8(const void* x, const float* gamma, const void* w_gate8, const float* w_gate_scale,
                                      const void* w_up8, const float* w_up_scale, const void* w_down8,
                                      const float* w_down_scale, void* out, int64_t tokens, int64_t hidden,
                                      int64_t intermediate, float eps, int x_dtype, int out_dtype, void* stream) {
  PTO_DISPATCH_LOCK();
  using namespace pto_hip;
  if (!ctx().initialized) return fail(PTO_HIP_ERR_NOT_INITIALIZED, "pto_hip_init has not been called");
  PTO_CHECK_ARG(tokens >= 0 && hidden > 0 && intermediate > 0, "ffn_fp8: bad shape T=%lld H=%lld I=%lld",
                (long long)tokens, (long long)hidden, (long long)intermediate);
  PTO_CHECK_ARG(tokens < (1 << 30) && hidden < (1 << 30) && intermediate < (1 << 30), "ffn_fp8: shape too large");
  if (tokens == 0) return PTO_HIP_OK;
  PTO_CHECK_ARG(x && w_gate8 && w_gate_scale && w_up8 && w_up_scale && w_down8 && w_down_scale && out,
                "ffn_fp8: null tensor pointer");
  PTO_CHECK_ARG(x_dtype == PTO_HIP_BF16 || x_dtype == PTO_HIP_FP16, "ffn_fp8: activation dtype %s not in {BF16, FP16}",
                dtype_name(x_dtype));
  PTO_CHECK_ARG(out_dtype == PTO_HIP_FP32 || out_dtype == x_dtype,
                "ffn_fp8: output dtype %s must be FP32 or the activation dtype %s", dtype_name(out_dtype),
                dtype_name(x_dtype));
  if (hidden % gemm8::BK != 0 || intermediate % gemm8::BK != 0)
    return fail(PTO_HIP_ERR_UNSUPPORTED, "ffn_fp8: hidden %lld and intermediate %lld must be multiples of %d",
                (long long)hidden, (long long)intermediate, gemm8::BK);
  PTO_CHECK_ARG(((uintptr_t)x | (uintptr_t)gamma | (uintptr_t)w_gate8 | (uintptr_t)w_up8 | (uintptr_t)w_down8 |
                 (uintptr_t)out | (uintptr_t)w_gate_scale | (uintptr_t)w_up_scale | (uintptr_t)w_down_scale) % 16 == 0,
                "ffn_fp8: operand and channel-scale pointers must be 16-byte aligned");
  // the row quantiser keeps a whole row in registers: refuse longer rows before anything is queued
  constexpr int64_t kMaxRow = (int64_t)8 * gemm8::kRowThreads * gemm8::kRowVecs;
  if (hidden > kMaxRow || intermediate > kMaxRow)
    return fail(PTO_HIP_ERR_UNSUPPORTED, "ffn_fp8: hidden %lld and intermediate %lld may be at most %lld (the per-row "
                "quantiser holds a row in registers)", (long long)hidden, (long long)intermediate, (long long)kMaxRow);
  hipStream_t st = (hipStream_t)stream;

  auto pad = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t x8_bytes = pad((size_t)tokens * hidden), h8_bytes = pad((size_t)tokens * intermediate);
  const size_t h_bytes = pad((size_t)tokens * intermediate * 2), s_bytes = pad((size_t)tokens * sizeof(float));
  void* ws = nullptr;
  int rc = workspace(x8_bytes + h8_bytes + h_bytes + 2 * s_bytes, &ws);
  if (rc) return rc;
  char* base = reinterpret_cast<char*>(ws);
  uint8_t* x8 = reinterpret_cast<uint8_t*>(base);
  uint8_t* h8 = reinterpret_cast<uint8_t*>(base + x8_bytes);
  void* h = base + x8_bytes + h8_bytes;
  float* sx = reinterpret_cast<float*>(base + x8_bytes + h8_bytes + h_bytes);
  float* sh = reinterpret_cast<float*>(base + x8_bytes + h8_bytes + h_bytes + s_bytes);

  // RMSNorm prologue and the activation quantiser are one row kernel
  rc = gemm8::row_quant(x, gamma, gamma != nullptr, x8, sx, tokens, hidden, eps, x_dtype, st);
  if (rc) return rc;

  gemm8::Params p1{};
  p1.a = x8;
  p1.b0 = reinterpret_cast<const uint8_t*>(w_gate8);
  p1.b1 = reinterpret_cast<const uint8_t*>(w_up8);
  p1.sa = sx;
  p1.sb0 = w_gate_scale;
  p1.sb1 = w_up_scale;
  p1.c = h;
  p1.lda = hidden;
  p1.ldb = hidden;
  p1.ldc = intermediate;
  p1.m = (int)tokens;
  p1.n = (int)intermediate;
  p1.k = (int)hidden;
  const bool bf16 = x_dtype == PTO_HIP_BF16;
  rc = bf16 ? gemm8::launch_tiles<true, __bf16>(p1, true, st) : gemm8::launch_tiles<true, _Float16>(p1, true, st);
  if (rc) return rc;
  if (p1.splits > 1) {
    // k split: the quantiser sums the slabs itself, h is not written
    const gemm8::SlabRows sl{p1.slabs, p1.sa, p1.sb0, p1.sb1, tokens * intermediate, p1.splits};
    if (bf16) gemm8::launch_row_quant<__bf16, false, true>(nullptr, nullptr, h8, sh, tokens, intermediate, 0.f, sl, st);
    else gemm8::launch_row_quant<_Float16, false, true>(nullptr, nullptr, h8, sh, tokens, intermediate, 0.f, sl, st);
    PTO_CHECK_HIP(hipGetLastError());
  } else {
    rc = gemm8::row_quant(h, nullptr, false, h8, sh, tokens, intermediate, 0.f, x_dtype, st);
    if (rc) return rc;
  }

  gemm8::Params p2{};
  p2.a = h8;
  p2.b0 = reinterpret_cast<const uint8_t*>(w_down8);
  p2.sa = sh;
  p2.sb0 = w_down_scale;
  p2.c = out;
  p2.lda = intermediate;
  p2.ldb = intermediate;
  p2.ldc = hidden;
  p2.m = (int)tokens;
  p2.n = (int)hidden;
  p2.k = (int)intermediate;
  if (out_dtype == PTO_HIP_FP32) return gemm8::launch_any<false, float>(p2, st);
  return x_dtype == PTO_HIP_BF16 ? gemm8::launch_any<false, __bf16>(p2, st)
                                 : gemm8::launch_any<false, _Float16>(p2, st);
}

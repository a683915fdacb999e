// Launch shapes chosen on the host from sizes alone (plain C++, no device code).
#pragma once

#include <algorithm>
#include <cstdint>

namespace pto_hip {

// Workgroups of a skinny projection (w8a16.hip): `slabs` output slabs of `ks` 32-row steps each, four wavefronts per
// workgroup with at least min_steps steps each, at most `most` workgroups (one per CU: a second one on some CUs is what
// the slowest CU waits for, 17 MB of codes take 8.2 us on 256 and 9.9 on 288).
// Where the slabs allow it a whole number of workgroups per slab, so that a workgroup has one run and its
// partial sums one slab (117 MB pair of codes at 32 rows: 224 workgroups 29 us, 256 33); of those the smallest number with
// the same count of rounds per wavefront.  Between 4/8 and 5/8 of the CUs one workgroup per slab would leave three CUs
// of eight without work, and even shares of the list over all of them win from 64 steps on, launch and finish at 1 / 32 rows:
// 5120 x 17408 16-bit (136 slabs) 41.9 / 51.4 -> 34.6 / 38.7 us, 4096 x 18432 (144) 34.3 / 41.4 -> 29.8 / 33.3, the pair 8192 x
// 10240 (160) 68.8 / 86.3 -> 61.1 / 64.8, int8 pairs 5120 x 17408 (136) 41.2 / 53.9 -> 36.2 / 45.2 and 2048 x 10240 (160) 16.8 / 20.8 ->
// 13.6 / 19.2; but 16-bit 4096 x 11008 (172) 35.1 / 40.8 -> 38.5 / 44.0, and with 48 steps int8 1536 x 8960 (140) 12.9 / 14.9 -> 12.0 / 16.0.
inline int64_t skinny_workgroups(int64_t slabs, int64_t ks, int64_t most, int64_t min_steps) {
  constexpr int64_t kWaves = 4;
  if (slabs > most) return most;
  if (slabs * 2 > most && slabs * 8 <= most * 5 && ks >= 64) return most;
  auto rounds = [&](int64_t per_slab) { return ((ks + per_slab - 1) / per_slab + kWaves - 1) / kWaves; };
  int64_t per_slab = std::max<int64_t>(1, std::min<int64_t>(most / slabs, ks / (kWaves * min_steps)));
  while (per_slab > 1 && rounds(per_slab - 1) == rounds(per_slab)) --per_slab;
  return slabs * per_slab;
}

// Tile height (64 * *height rows, 0: the 256-row tile with eight wavefronts) and k split count of a product with 16-bit
// weights: the pair with the least estimated time in microseconds.  Timed against every pair (with its finish launch) at 33
// to 4000 rows of eighteen weight shapes, 1024 x 3072 to 8192 x 22016, the one it picks is slower than the best by
// 1.0 % on average and 23 % at most in gate/up passes, by 2.3 % and 20 % in single ones.  Whole rounds of
// workgroups over the CUs cost (a + b) ns per k row a workgroup walks, a last partial one a + b * its share of the CUs -
// L2 and the clock are shared -, each round c more for its start and its stores; not less than the weights take to
// stream; a split the finish launch and the slabs' way out and back, dearer once they outgrow the last-level cache.
// The 256-row form with a ragged last row tile keeps 80 registers in scratch in the single-operand
// pass, which slows its slab stores (4096 x 4096 at 400 rows 50 us, 34 with eight wavefronts): there the eight-wavefront
// form is a candidate too, where its loop is the direct one the costs were taken from (n and k in whole tiles).  With ragged columns or k
// the 256-row form always keeps them and that loop is never ahead (at 33 to 1800 rows of fourteen such weight shapes, every tile and split timed, its best is
// behind the best of the four-wavefront forms in all 230 passes): there it is dearer by what was measured beside its cost, 1.1 times up to
// two rounds and 1.2 with slabs.  8192 x 8128 at 400 / 900 rows 99 / 151 -> 73 / 121 us, 8192 x 7232 90 / 141 -> 68 / 114.
// Over several rounds the 256-row tile, with the fewest operand bytes per MFMA, is ahead of what its one-round costs say
// (back to back, 256 / 192 rows a tile: gate/up 5120 x 13824 at 1800 rows 506 / 528 us, 8192 x 22016 at 3000 1816 / 1846,
// 4096 x 10752 at 2709 417 / 454): it wins unless another is 5 % ahead.  At 0.97 instead of 0.95 the first two are lost, at
// 0.93 others are (4096 x 14336 at 3000 rows by 5 %).
// Up to 64 rows a single matrix is bound by its stream, and splits that start a multiple of 8 MiB apart ask the same memory
// channels at the same time: 11008 x 4096 in 11 splits of 1024 k rows 31.4 us, in 16 of 704 26.5; 14336 x 4096 in 14 of
// 1024 33.3, in 16 of 896 31.3.
// `forced`: height given, only the split count is chosen.
// Returns the estimate (without the launch's own time).
inline double choose_quad(int m, int n, int k, bool dual, int64_t num_cu, int forced, int* height, int* want) {
  constexpr int BK = 64, BN = 256, kMaxSplits = 16;
  struct Cost {
    double a, b, c;
  };
  // [0]: eight wavefronts
  static constexpr Cost kCost[5] = {{16.84, 7.88, 2.31}, {5.8, 6.58, 2.03}, {10.02, 5.93, 2.83}, {12.72, 5.69, 4.69}, {16.16, 8.28, 3.52}};
  const double weights_mb = (double)k * n * (dual ? 2 : 1) * 2e-6;
  const bool spills = !dual && (n % BN != 0 || k % 32 != 0);  // the 256-row form, whatever m
  double best = 1e30;
  for (int h = 0; h <= 4; ++h) {
    if (forced ? h != forced : (h == 0 && (dual || m % 256 == 0 || k % BK != 0 || n % BN != 0))) continue;
    const int bm = h ? 64 * h : 256;
    const int bn = dual ? BN / 2 : BN;
    const int64_t tiles = (int64_t)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
    for (int s = 1; s <= kMaxSplits; ++s) {
      if (s > 1 && k < 4 * BK * s) break;
      const int64_t kps = ((k + s * BK - 1) / (s * BK)) * BK;
      if ((k + kps - 1) / kps != s) continue;
      const int64_t full = tiles * s / num_cu, left = tiles * s % num_cu;
      const Cost& q = kCost[h];
      double t = (double)kps * 1e-3 * ((double)full * (q.a + q.b) + (left ? q.a + q.b * (double)left / (double)num_cu : 0.0)) +
                 q.c * (double)(full + (left ? 1 : 0));
      t = std::max(t, weights_mb / 10.2);
      if (s > 1) {
        const double slab_mb = (double)s * m * n * (dual ? 2 : 1) * 4e-6;
        t += 2.95 + slab_mb * (dual ? 0.177 : 0.374) + std::max(slab_mb - 128.0, 0.0) * 0.29;
        if (!dual && m <= 64 && kps * n % (4 << 20) == 0) t *= 1.05;
      }
      if (h == 4 && full >= 2) t *= 0.95;
      else if (h == 4 && spills) t *= 1.1;
      if (h == 4 && spills && s > 1) t *= 1.2;
      if (t < best) {
        best = t;
        *height = h;
        *want = s;
      }
    }
  }
  return best;
}

// Tile of the small-call form (narrow_gemm.h) for a product with 16-bit weights: 1: 16 rows x 32 channels, 2: 32 x 32, 3: 32 x 64, 4: 64 x 64;
// 0: the tiled GEMM.  Estimated microseconds, fitted to 40 to 1024 rows of nineteen weight shapes from 512 x 512 to 2048 x 5632
// (rms 5 to 11 %): a launch, the operand KB of a tile once per round of workgroups over the CUs, and what the weights take to
// arrive.  tiled_us: choose_quad's estimate, which takes 1.11 of itself and 2 us in the same measure; the form has to be 5 % ahead.  Over the
// 175 products of 33 and more rows among them the estimate was 1.35 times as fast as the tiled GEMM, the best of all tiles and forms 1.38.  Timed alone: in a
// block the activations of the down projection have just been written by other XCDs, and every tile of channels fetches them again.  Hence
// the last term, 1.3 us per MB of a single product's activations: without it blocks of 333 to 1000 rows lost up to 17 % (768 x 2560 at 768 rows 25.7
// -> 30.2 us, 1024 x 3072 at 640 30.3 -> 35.4).  With it, over 110 blocks of 64 to 1300 rows of
// ten shapes, 512 x 1024 to 1280 x 4096: 1.13 times as fast as the tiled form, five slower, by 2 to 4 %.
// Three corrections from 470 blocks of 33 to 1400 rows, 512 to 2300 wide, channels in eights and in 64s (kernel traces, products one by one): a
// single tiled product with two or three k splits takes 2 us less than choose_quad says; rows that are no multiple of 64 channels put every
// piece of a pair's weights on a line more, 0.005 us a KB; and 64 x 64 tiles wait for a pair's weights beyond 8 MB, 0.3 us a MB.  Blocks slower than
// on the tiled form alone by more than 1 %: 23 -> none (65 rows of 1216 x 4408 31.1 -> 28.0 us, 195 of 1096 x 3680 35.0 -> 31.2, 232 of 1152 x
// 4032 32.3 -> 30.2, 733 of 1024 x 2176 31.8 -> 30.5).
// Up to 32 rows a product in the skinny form streams its weights once, in two launches; this form is ahead up to 1.6 million weights
// (us, skinny -> this, 1 / 32 rows: 512 x 1024 pair 6.1 / 7.3 -> 4.2 / 4.5, 1024 x 1024 5.7 / 7.3 -> 4.1 / 4.7, 2048 x 768 6.1 / 7.5 ->
// 5.6 / 6.8; but 768 x 2048 pair 7.0 / 8.4 -> 7.7 / 7.7, 1024 x 2048 pair 7.0 / 8.6 -> 9.3 / 9.5).
inline bool narrow_beats_skinny(int64_t k, int64_t n, bool dual) { return k * n * (dual ? 2 : 1) <= 1600000; }

// splits: of k, with which the tiled form would run.
inline int choose_narrow(int64_t m, int64_t n, int64_t k, bool dual, int64_t num_cu, double tiled_us, int splits = 1) {
  struct Tile {
    int rows, channels;
    double us[2], round[2], mb[2];  // of a single product and of a pair
  };
  static constexpr Tile kTiles[4] = {{16, 32, {2.31, 2.40}, {0.0171, 0.0154}, {0.394, 0.371}},
                                     {32, 32, {2.33, 2.22}, {0.0201, 0.0226}, {0.313, 0.274}},
                                     {32, 64, {1.83, 1.67}, {0.0226, 0.0257}, {0.070, 0.084}},
                                     {64, 64, {2.80, 2.77}, {0.0191, 0.0275}, {0.165, 0.0}}};
  double best = (1.112 * tiled_us + 2.05 - (!dual && (splits == 2 || splits == 3) ? 1.9 : 0.0)) * 0.95;
  int tile = 0;
  for (int i = 0; i < 4; ++i) {
    const Tile& t = kTiles[i];
    const int64_t wgs = ((m + t.rows - 1) / t.rows) * ((n + t.channels - 1) / t.channels);
    const double kb = (double)k * 2.0 * (t.channels * (dual ? 2 : 1) + t.rows) * 1e-3;
    const double weights_mb = (double)k * n * (dual ? 2 : 1) * 2e-6;
    const double round = t.round[dual] + (dual && n % 64 != 0 ? 0.005 : 0.0);
    double us = t.us[dual] + round * (double)((wgs + num_cu - 1) / num_cu) * kb + t.mb[dual] * weights_mb;
    if (!dual) us += 1.3 * (double)m * k * 2e-6;
    else if (i == 3) us += 0.3 * std::max(weights_mb - 8.0, 0.0);
    if (us < best) {
      best = us;
      tile = i + 1;
    }
  }
  return tile;
}

// Tile of the small-call form of e4m3 products (narrow_gemm8.h): 1: 16 rows x 16 channels, 2: 32 x 32, 3: 64 x 32; 0: the tiled GEMM.
// Estimated microseconds, fitted to 1 to 1024 rows of sixteen weight shapes from 512 x 1024 to 13824 x 5120 (rms 10 to 19 %): a launch, the operand
// KB of a tile once per round of workgroups over the CUs, and what the weights take to arrive.  tiled_us: what the tiled form's own
// estimate says; this form has to be 5 % ahead.  Timed at other row counts, and with six other weight shapes among them, the rule is 1.45 times as
// fast as the tiled form alone, the best of all four 1.48, and nothing is slower by more than the noise of 2 %.
inline int choose_narrow8(int64_t m, int64_t n, int64_t k, bool dual, int64_t num_cu, double tiled_us) {
  struct Tile {
    int rows, channels;
    double us[2], round[2], kb[2], mb[2];  // of a single product and of a pair
  };
  static constexpr Tile kTiles[3] = {{16, 16, {1.78, 1.83}, {0.39, 1.68}, {0.0306, 0.0057}, {0.0, 0.170}},
                                     {32, 32, {1.36, 2.61}, {0.72, 1.02}, {0.0286, 0.0219}, {0.0, 0.111}},
                                     {64, 32, {0.0, 1.56}, {5.09, 0.64}, {0.0198, 0.0361}, {0.0, 0.0}}};
  double best = 0.95 * tiled_us;
  int tile = 0;
  for (int i = 0; i < 3; ++i) {
    const Tile& t = kTiles[i];
    const int64_t wgs = ((m + t.rows - 1) / t.rows) * ((n + t.channels - 1) / t.channels);
    const double kb = (double)k * (t.channels * (dual ? 2 : 1) + t.rows) * 1e-3;
    const double us = t.us[dual] + (double)((wgs + num_cu - 1) / num_cu) * (t.round[dual] + t.kb[dual] * kb) + t.mb[dual] * (double)k * n * (dual ? 2 : 1) * 1e-6;
    if (us < best) {
      best = us;
      tile = i + 1;
    }
  }
  return tile;
}

// Whether a projection of m rows inside a decoder layer or block streams its weights (stream_rows.h) instead of running as a tiled GEMM.
// Measured in whole layers with each projection switched, 36 / 56 / 80 / 96 rows of twelve models from 1024 x 3072 to 8192 x 28672, us gained:
// 16-bit weights: pairs from 30 million on (4096 x 14336 4 / 5 / 4 / 6, 3072 x 8192 9 / 14 / 13 / 14, 8192 x 16384 10 / 10 / 11 / 12; 2048 x 5632, 23 million,
// lost 1 / 2 / 4 / 4), deep single ones from 40 million on (14336 x 4096 7 / 10 / 9 / 11, 13824 x 5120 9 / 11 / 10 / 9; 8192 x 3072 lost 2 to 6,
// square ones 0 to 7).
// int8: pairs from 80 million on (4096 x 14336 10 / 9 / 7 / 4, 4096 x 11008 11 / 8 / 6 / 6; 3072 x 8192 lost 0 to 3), deep single ones of 5120 channels
// and 60 million up, with few slabs a channel (13824 x 5120 3 / 3 / 2 / 2, 16384 x 8192 7 / 5 / 4 / 3; 14336 x 4096 lost 0 to 2).
// Few k, up to 64 rows (layers with these projections tiled -> streamed, k split in both, 36 / 48 / 64 rows, us gained): hidden 1024 5 / 4 / 2,
// 1280 4 / 3 / 0, 1536 4 / 2 / -1, 1792 2 / 1 / 0, 2048 2 / 1 / 0, 2304 2 / 1 / 0, 3072 3 / 2 / 2, 3584 8 / 9 / 8.
// Why k from 1280 to 3072 stays tiled above 48 rows: the two are level there, or streams behind, where a product has whole tiles of 256 channels and as
// many k splits streamed as tiled, k / 256 (layers, tiled -> streamed, us: 64 rows of 2048 67.1 -> 67.2, of 2304 70.6 -> 70.6; 61 of 1856 with 4608 q/k/v
// channels 76.7 -> 77.7, 60 of 2368 with 1536 73.4 -> 73.7).  Few k leave the tiled form few splits and most CUs idle; many k give it more of them than
// the CUs hold of the streamed form's, and so more partial sums (64 rows of 3072 87.8 -> 84.3, of 4096 107.1 -> 102.1).  Streams would also be ahead in between where n ends
// inside a tile or the CUs hold fewer streamed splits (60 rows of 2112 with 1152 q/k/v channels 69.0 -> 67.2, 58 of 2688 with 4608 96.4 -> 93.2): not used.
// A pair of more slabs than half the CUs has no k split, and the fewer slabs beyond, the more CUs have none while the launch lasts as long as with 256.  Up to
// 2/3 of the CUs such pairs lose against the tiled GEMM: with 16-bit weights 1 to 7 us (36 / 48 / 57 / 64 / 80 / 96 rows of 4096 x 8960 3 / 4 / 5 / 4 / 4 / 4, 4992 x 9472 3 /
// 4 / 6 / 4 / 2 / 2, 52 of 3200 x 9216 3), unless the down projection streams as well, which only a streamed pair leaves its activations to (4096 x 9984 gains 4 / 5 /
// 3 / 3 / 0 / 0 in both), or k is below 2560 (45 x 2112 x 8320 7 gained); with int8 above 48 rows up to 0.6 of the CUs and above 64 rows up to 2/3 (4992 x 8960
// 1 and 1 gained, 3 / 3 / 5 / 5 lost, 4096 x 10496 7 / 7 / 2 / 4 gained, 2 / 1 lost), but not with a last slab that is no whole 128 channels, which the
// tiled int8 GEMM is slower with (65 to 96 rows of 4224 x 9664 gain 6 to 9).
constexpr int kStreamRowsMax = 96;
// k splits of a streamed projection: what the CUs hold of its 128-channel slabs, of at least eight 32-row steps each.
inline int stream_splits(int64_t k, int64_t n, bool dual, int64_t num_cu) {
  const int64_t slabs = (n + 127) / 128 * (dual ? 2 : 1), ks = (k + 31) / 32;
  return (int)std::max<int64_t>(1, std::min<int64_t>(num_cu / slabs, ks / 8));
}
inline bool stream_rows_ahead(int64_t m, int64_t k, int64_t n, bool dual, bool w16, int64_t num_cu) {
  const int64_t weights = k * n * (dual ? 2 : 1), slabs = (n + 127) / 128 * (dual ? 2 : 1);
  if (dual && 2 * slabs > num_cu && 3 * slabs < 2 * num_cu) {
    if (w16 && k >= 2560 && !(weights >= 80000000 && n >= 2 * k)) return false;
    if (!w16 && n % 128 == 0 && m > 48 && (m > 64 || 5 * slabs < 3 * num_cu)) return false;
  }
  if (w16) return dual ? weights >= 30000000 : weights >= 40000000 && k >= 2 * n;
  if (dual) return weights >= 80000000 || (m <= 64 && k <= (m <= 48 ? 1536 : 1280));
  return (m <= 64 && k <= 4096 && (m <= 48 || k <= 1280 || k >= 3072)) || (n >= 5120 && weights >= 60000000 && k >= 2 * n);
}

// Row a workgroup takes where one writes a row of the blocked layout [K/8][rows][8]: its 128-byte lines are eight rows' pieces, and
// eight rows whose workgroups run on one XCD (workgroup id mod 8) meet in that XCD's L2.  Of every 64 ids the first groups * 8, groups being the
// whole groups of eight rows there, go XCD by XCD to the groups one after the other: eight groups have an XCD each, fewer (`groups` ids
// an XCD) ceil(8 / groups) or one more, where rows as they come have all eight (as they had at 40 to 47 and 56 to 63 rows when ids were dealt to
// the groups in turn: layer of 56 sequences, int8, 4096 wide 112.5 -> 111.4 us, block of 60 tokens 4096 x 11008 71.8 -> 71.0).  A permutation of 0 .. rows - 1; rows 0, for up to 32 rows, where
// nothing is gained: as they come.
constexpr int blocked_row(int id, int rows) {
  if (rows == 0) return id;
  const int base = id & ~63, at = id & 63, groups = (rows - base < 64 ? rows - base : 64) >> 3;
  return at < groups * 8 ? base + (at & 7) * groups + (at >> 3) : id;
}

// Tokens per context partition of a workgroup-form attention launch (a workgroup per (sequence, KV head) pair, its
// wavefronts take the partitions) over an e4m3 cache at head_dim 128; `plain` is the rule for 16-bit caches, two wavefronts per
// CU and at most 2048 tokens.  A chunk of codes is half the bytes of a 16-bit one, so two wavefronts do not keep enough requests in
// flight, and a partition of 2048 tokens is what the launch waits for when lengths are ragged: from tables of more than 1536
// tokens on four wavefronts per CU, partitions of equal length: of 512 to 1024 tokens but for whole blocks (416 of a 1568-token table of 32-token
// ones) and max_parts (1536 of a 12000-token table).  Attention call, us, tables for
// (pairs x tokens) with equal / ragged lengths: 256 x 4096 63.0 / 61.4 -> 42.6 / 34.4, 320 x 2200 49.9 / 48.0 -> 34.1 / 30.0, 768 x 3000
// 120 / 70.4 -> 98 / 69; but one partition split, 1024 x 1400 56.2 -> 59.7, hence 1536.  16-bit caches are the other way round: 768 x 3000 113.9 ragged
// -> 119, 256 x 4096 equal 80.7 -> 82.6.  The plain rule stays where its own wavefronts fill the CUs as well, lengths equal / down to half / to a tenth:
// from four partitions on (plain -> more: 320 x 8000 108 / 85 / 79 -> 119 / 100 / 78), between 4.5 and 6 times 2048 tokens per CU (448 x 6000
// 115 / 92 / 82 -> 117 / 100 / 85, 1024 x 2600 114 / 92 / 77 -> 118 / 96 / 81; below they are ahead with ragged lengths, 512 x 3500
// 81 / 72 / 66 -> 78 / 65 / 51, 768 x 3000 100 / 84 / 73 -> 106 / 88 / 68, and above, 1600 x 3500 263 / 198 / 159 -> 250 / 190 / 149), and for one partition of four pairs per CU (1600 x 2000 143 / 119 / 96 -> 150 / 119 / 92).
// Not more partitions than a workgroup has wavefronts (max_parts: the form needs no scratch), nor than whose partials, should the grid
// form be taken after all, fit the fixed area of the entry point that allocates nothing.
inline int64_t attn_e4m3_partition_tokens(int64_t pairs, int64_t max_ctx, int64_t num_cu, int64_t max_parts, int64_t bytes_per_part,
                                          int64_t scratch, int64_t plain) {
  if (max_ctx <= 1536) return plain;
  const int64_t before = (max_ctx + plain - 1) / plain, load = pairs * max_ctx / 2048;
  if (before >= 4 || (2 * load > 9 * num_cu && load < 6 * num_cu) || (before == 1 && pairs >= 4 * num_cu)) return plain;
  const int64_t want = std::max<int64_t>(1, (4 * num_cu + pairs - 1) / pairs);
  const int64_t tokens = std::min<int64_t>(1024, std::max<int64_t>(512, (max_ctx + want - 1) / want));
  int64_t parts = std::min((max_ctx + tokens - 1) / tokens, max_parts);
  parts = std::min(parts, scratch / bytes_per_part);
  if (parts <= before) return plain;
  return (max_ctx + parts - 1) / parts;
}

// What partition lengths are multiples of: the KV block (`block`, or its part that divides a long one) or a half, quarter ... of it down to 64
// tokens.  A launch of a few pairs is a chain - table, first rows, a chunk of 32 tokens after the other - that halves are two
// chunks shorter than whole 128-token blocks; what they cost is another partial per query row (written, read by the merge) and, from one
// partition to two, the merge itself.  So a partition is halved as far as the wavefronts it gives leave that hidden, by the `weight` of a partial beside its
// part of the cache: query rows per KV head (`rows`, as far as one wavefront carries them) against the length, squared since a short
// partition is also the shorter chain.  Measured against whole blocks and every halving at 2 to 250 pairs, tables of 1 to 24
// blocks of 128, 256 and 512 tokens, 1 to 64 query heads per KV head, equal and ragged lengths (3828 calls, whole blocks -> this rule):
// -14.1 % on average, 27 calls more than 3 % slower, by 6 % at most; 0.8 % behind the best of each.  Us, whole blocks -> halved:
// one partition: 64 pairs x 384 of a 512-token block, 16 heads 14.1 -> 12.5, quarters 9.1, but 8 x 96 of a 128-token block 6.1 -> 6.9 (kept whole);
// above a pair per CU 300 x 512 of one block 21.6 -> 18.4, e4m3 18.0 -> 15.5, but of a 128-token one 8.1 -> 7.9 and 16-bit head_dim 256 29.9 -> 33.8;
// two, the four of which a workgroup's wavefronts can merge (head_dim 256 with few heads only as far as CUs idle): 160 x 224, 16 heads 9.2 -> 8.0;
// more: 8 x 1504, 16 heads 10.7 -> 9.8; but 96 x 480, 32 heads 12.2 -> 19.6, 8 heads at head_dim 256 16.2 -> 18.7 (kept whole).
// Halves as long as the table's blocks gave fewer than two wavefronts per CU, whatever the rows, as before: -11.1 % on average, 729 calls more than
// 3 % slower, by up to 88 %.
// `wg_parts` > 0: the workgroup form is asked for, which up to that many partitions stay within.  bytes_per_part, scratch: as above.
inline int64_t attn_partition_align(int64_t pairs, int64_t max_ctx, int64_t block, int64_t num_cu, int64_t bytes_per_part, int64_t scratch,
                                    int64_t rows = 1, int64_t head_dim = 128, bool e4m3 = false, int64_t wg_parts = 0) {
  const bool long_rows = head_dim * (e4m3 ? 1 : 2) > 256;  // of the cache: more of the time is its stream
  const bool short_rows = e4m3 && head_dim == 128 && rows <= 16;
  int64_t align = block;
  for (int64_t len = block; len >= 128 && len % 64 == 0; len /= 2) {
    const int64_t parts = (max_ctx + len - 1) / len;
    if (2 * parts * bytes_per_part > scratch || (parts <= wg_parts && 2 * parts > wg_parts)) break;
    const double weight = (double)(rows * head_dim) / 128.0 * (128.0 / (double)len) * (128.0 / (double)len);
    int quarters;  // wavefronts up to which a partition is halved, in quarters of the CUs
    if (parts == 1) quarters = weight > 4.0 ? 0 : weight > 1.0 || len <= 128 || long_rows ? 4 : e4m3 ? 7 : 6;
    else if (parts == 2) quarters = long_rows && rows < 8 && len <= 128 ? 3 : 8;
    else if (parts <= 4 && short_rows) quarters = 8;  // (eight of which a workgroup can merge)
    else if (weight >= 16.0) quarters = short_rows ? 3 : 2;
    else if (weight > 4.0) quarters = e4m3 && rows <= 8 ? 4 : 3;
    else if (len <= 128) quarters = short_rows ? 6 : long_rows ? 3 : 4;
    else if (long_rows) quarters = 4;
    else quarters = weight > (e4m3 ? 2.0 : 1.0) ? 5 : short_rows && weight <= 1.0 ? 8 : 6;
    if (pairs * parts * 4 <= quarters * num_cu && pairs * parts < 2 * num_cu) align = len / 2;
    else if (parts > 1) break;  // (one partition: four can still be ahead where two are not)
  }
  return align;
}

}  // namespace pto_hip

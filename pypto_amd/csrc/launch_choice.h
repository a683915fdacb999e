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

}  // namespace pto_hip

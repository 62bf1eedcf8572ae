// Reverse of one RK3 stage (famrdp_reverse.hip, its own translation unit):
// the viscous reverse beside the i and k axes, then the j axis and the rest of
// each cell, over the plan's adjoint block table.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "famrdp_kernels.h"

namespace famrdp {

// One wave's share of a sweep along an axis: cells p0 .. p1-1 of it, over the
// SWEEP_IK plane cells (i sweep: lanes 3 .. 60 of the wave), SWEEP_J columns
// (j sweep: all lanes) or SWEEP_V cells of the plane with extended rows
// (viscous part: lanes 2 .. 61) from base on.
struct SweepTile {
  int32_t block, p0, p1, base;
};
constexpr int SWEEP_IK = 58, SWEEP_J = 64, SWEEP_V = 60;
constexpr int SWEEP_WAVES = 2;   // waves of a sweep that a SIMD holds (registers)

// What a sweep runs over: per block its cells along the swept axis and across
// it, `lanes` of the latter a wave.
struct SweepSet {
  std::vector<int32_t> along, across;
  int lanes;
  int64_t waves(int len) const {
    int64_t n = 0;
    for (size_t b = 0; b < along.size(); ++b)
      n += (int64_t)((across[b] + lanes - 1) / lanes) * ((along[b] + len - 1) / len);
    return n;
  }
};

// The sweep length of the sets that share a launch on a GPU that holds `slots`
// waves at once.  A wave sweeps len cells and about SWEEP_EXTRA more around
// them: the least (rounds of waves) x (len + SWEEP_EXTRA).  Short sweeps fill
// a GPU that a small block would leave idle (36^3: length 1, 37 us a stage;
// 3: 54 us), long ones waste less on their ends (100^3: 20 for the two sweeps
// along i together, 133 us; 10: 140 us).
constexpr int SWEEP_EXTRA = 5, SWEEP_MAX = 64;
inline int sweep_len(const std::vector<const SweepSet*>& sets, int64_t slots) {
  int best = 1;
  int64_t best_cost = 0;
  for (int len = 1; len <= SWEEP_MAX; ++len) {
    int64_t n = 0;
    for (const SweepSet* s : sets) n += s->waves(len);
    const int64_t cost = (n + slots - 1) / slots * (len + SWEEP_EXTRA);
    if (len == 1 || cost < best_cost) {
      best = len;
      best_cost = cost;
    }
  }
  return best;
}

// The table of a set at length len: a block's cells along the axis are split
// evenly.
inline std::vector<SweepTile> sweep_tiles(const SweepSet& s, int len) {
  std::vector<SweepTile> t;
  for (size_t b = 0; b < s.along.size(); ++b) {
    const int nseg = (s.along[b] + len - 1) / len;
    for (int g = 0; g < nseg; ++g)
      for (int32_t c = 0; c < s.across[b]; c += s.lanes)
        t.push_back(SweepTile{(int32_t)b, (int32_t)((int64_t)g * s.along[b] / nseg),
                              (int32_t)((int64_t)(g + 1) * s.along[b] / nseg), c});
  }
  return t;
}

void launch_stage_vjp(const BlockDesc* blocks, const SweepTile* sv, int nv, const SweepTile* sik, int nik,
                      const SweepTile* sj, int nsj, int stage, const Gas& gas, double dt, int lim, hipStream_t st);

}  // namespace famrdp

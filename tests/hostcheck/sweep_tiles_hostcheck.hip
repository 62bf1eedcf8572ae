// Test-only host build of the reverse sweeps' tables
// (famrdp-jax_amd/csrc/famrdp_reverse.h).  Never loaded by the product.
#include "famrdp_reverse.h"

using namespace famrdp;

extern "C" {

// The table of nb blocks; returns its length, or -1 if it exceeds cap.
int sweep_table(int nb, const int32_t* along, const int32_t* across, int lanes, int64_t slots, int cap, int32_t* out) {
  const SweepSet s{std::vector<int32_t>(along, along + nb), std::vector<int32_t>(across, across + nb), lanes};
  const std::vector<SweepTile> t = sweep_tiles(s, sweep_len({&s}, slots));
  if ((int)t.size() > cap) return -1;
  for (size_t i = 0; i < t.size(); ++i) {
    out[4 * i] = t[i].block;
    out[4 * i + 1] = t[i].p0;
    out[4 * i + 2] = t[i].p1;
    out[4 * i + 3] = t[i].base;
  }
  return (int)t.size();
}

}

// Test-only host build of the choice of a stage-kernel variant
// (famrdp-jax_amd/csrc/famrdp_tune.h) with timings made up.
#include "famrdp_tune.h"

extern "C" int hc_tune(int nv, const bool* fits, int reps, const float* cold, const float* warm, const float* more,
                       float* ms) {
  int best = -1;
  auto first = [&](int v, float& a, float& b) { a = cold[v]; b = warm[v]; return 0; };
  auto rest = [&](int v, int, float& t) { t = more[v]; return 0; };
  famrdp::tune_variants(nv, fits, reps, first, rest, ms, best);
  return best;
}

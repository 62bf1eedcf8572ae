// Choice of the stage-kernel variant from timings (famrdp_plan_autotune).
// Host code, so that it can be checked with timings made up.
#pragma once

#include <algorithm>

namespace famrdp {

// first(v, a, b): ms of two successive launch pairs of variant v, the first of
// them cold; rest(v, n, ms): ms of one of n more; both return nonzero on an
// error.  Every variant that fits runs two pairs, those within 1.5 of the best
// reps - 1 more.  The better of the two counts: one disturbed pair (the only one
// that was timed, once) must not drop the best variant.  Ties (within 1.5 %:
// stages 1 and 2 rank variants that close only to about that) keep the earlier
// variant.  ms: per variant, 1e30 for those that do not fit.
template <class First, class Rest>
int tune_variants(int nv, const bool* fits, int reps, First&& first, Rest&& rest, float* ms, int& best) {
  float least = 1e30f;
  for (int v = 0; v < nv; ++v) {
    ms[v] = 1e30f;
    if (!fits[v]) continue;
    float a = 0.f, b = 0.f;
    if (const int rc = first(v, a, b)) return rc;
    ms[v] = std::min(a, b);
    least = std::min(least, ms[v]);
  }
  best = 0;
  float best_ms = 1e30f;
  for (int v = 0; v < nv; ++v) {
    if (reps > 1 && ms[v] <= 1.5f * least) {
      float more = 0.f;
      if (const int rc = rest(v, reps - 1, more)) return rc;
      ms[v] = (ms[v] + more * (reps - 1)) / reps;
    }
    if (ms[v] < best_ms * 0.985f) { best_ms = ms[v]; best = v; }
  }
  return 0;
}

}  // namespace famrdp

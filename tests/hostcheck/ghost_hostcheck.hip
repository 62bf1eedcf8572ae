// Test-only host build of the ghost table (famrdp-jax_amd/csrc/famrdp_ghost.h):
// builds the table of a configuration and applies it to host arrays the way
// the two launches do, each launch's entries in ascending or descending order
// (on the GPU they run in any order).  Never loaded by the product.
#include "famrdp_ghost.h"

using namespace famrdp;

namespace {
void value(double* const* q, const std::vector<int64_t>& N, const GhostTable& t, int sb, int sc, int chain, double g,
           double R, double out[5]) {
  for (int v = 0; v < 5; ++v) out[v] = sb >= 0 ? q[sb][v * N[sb] + sc] : 0.0;
  const GhostChain& c = t.chains[chain];
  for (int i = 0; i < c.n; ++i) bc_apply(t.ops[c.op[i]], g, R, out);
}
}  // namespace

extern "C" {

// dims [nb][3]; cuts [ncut][4] target block, face, source block, face; bcs
// [nbc][3] block, face, kind with T_wall [nbc] and q_inf [nbc][5]; q [nb]
// pointers.  counts: direct, staged, late entries.
void ghost_apply(int nb, const int32_t* dims, int ncut, const int32_t* cuts, int nbc, const int32_t* bcs,
                 const double* T_wall, const double* q_inf, double g, double R, int reverse, double* const* q,
                 int32_t* counts) {
  const int G = 2;
  GhostTable t(G, nb, dims);
  std::vector<int64_t> N;
  for (int b = 0; b < nb; ++b) N.push_back((int64_t)dims[3 * b] * dims[3 * b + 1] * dims[3 * b + 2]);
  for (int c = 0; c < ncut; ++c) {
    const int32_t* x = cuts + 4 * c;
    const int32_t *dt = dims + 3 * x[0], *ds = dims + 3 * x[2];
    const int at = x[1] / 2, as = x[3] / 2;
    int e[3] = {dt[0], dt[1], dt[2]}, lt[3] = {0, 0, 0}, ls[3] = {0, 0, 0};
    e[at] = G;
    lt[at] = x[1] % 2 == 0 ? 0 : dt[at] - G;
    ls[as] = x[3] % 2 == 0 ? G : ds[as] - 2 * G;
    for (int a = 0; a < e[0]; ++a)
      for (int b = 0; b < e[1]; ++b)
        for (int k = 0; k < e[2]; ++k)
          t.copy(x[0], lt[0] + a, lt[1] + b, lt[2] + k, x[2],
                 (int32_t)(((int64_t)(ls[0] + a) * ds[1] + ls[1] + b) * ds[2] + ls[2] + k));
  }
  std::vector<BcEntry> byface[6];
  int64_t maxc[6] = {0, 0, 0, 0, 0, 0};
  for (int i = 0; i < nbc; ++i) {
    BcEntry e{bcs[3 * i], bcs[3 * i + 1], bcs[3 * i + 2], 0, T_wall[i], {}};
    for (int v = 0; v < 5; ++v) e.q_inf[v] = q_inf[5 * i + v];
    byface[e.face].push_back(e);
  }
  t.boundary(byface, maxc, false);
  t.finish();
  counts[0] = t.ndirect; counts[1] = t.nstaged; counts[2] = t.nlate;
  std::vector<double> stage((size_t)5 * t.nstaged);
  const int n1 = t.ndirect + t.nstaged, n2 = t.nstaged + t.nlate;
  for (int r = 0; r < n1; ++r) {
    const int i = reverse ? n1 - 1 - r : r;
    const GhostEntry& e = t.entries[i];
    double x[5];
    value(q, N, t, e.sb, e.sc, e.chain, g, R, x);
    for (int v = 0; v < 5; ++v) {
      if (i < t.ndirect) q[e.tb][v * N[e.tb] + e.tc] = x[v];
      else stage[(size_t)v * t.nstaged + (i - t.ndirect)] = x[v];
    }
  }
  for (int r = 0; r < n2; ++r) {
    const int i = reverse ? n2 - 1 - r : r;
    const GhostEntry& e = t.entries[t.ndirect + i];
    double x[5];
    if (i < t.nstaged) for (int v = 0; v < 5; ++v) x[v] = stage[(size_t)v * t.nstaged + i];
    else value(q, N, t, e.sb, e.sc, e.chain, g, R, x);
    for (int v = 0; v < 5; ++v) q[e.tb][v * N[e.tb] + e.tc] = x[v];
  }
}

}

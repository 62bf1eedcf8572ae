// Test-only host build of the ghost table's other two uses: a step from one set
// of arrays into another (every entry from the sources, the kept ones too) and
// the values recorded for the reverse sweep beside the first launch's entries.
// Never loaded by the product.
#include "famrdp_ghost.h"

using namespace famrdp;

namespace {

constexpr int G = 2;

struct Table {
  GhostTable t;
  std::vector<int64_t> N;
  double g, R;

  // dims [nb][3]; cuts [ncut][4] target block, face, source block, face; bcs
  // [nbc][3] block, face, kind with T_wall [nbc] and q_inf [nbc][5]
  Table(int nb, const int32_t* dims, int ncut, const int32_t* cuts, int nbc, const int32_t* bcs, const double* T_wall,
        const double* q_inf, double g_, double R_, const int64_t (&maxc)[6], bool snap)
      : t(G, nb, dims), g(g_), R(R_) {
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
    for (int i = 0; i < nbc; ++i) {
      BcEntry e{bcs[3 * i], bcs[3 * i + 1], bcs[3 * i + 2], 0, T_wall[i], {}};
      for (int v = 0; v < 5; ++v) e.q_inf[v] = q_inf[5 * i + v];
      byface[e.face].push_back(e);
    }
    t.boundary(byface, maxc, snap);
    t.finish();
  }
  void value(double* const* q, int sb, int sc, int chain, double out[5]) const {
    for (int v = 0; v < 5; ++v) out[v] = sb >= 0 ? q[sb][v * N[sb] + sc] : 0.0;
    const GhostChain& c = t.chains[chain];
    for (int i = 0; i < c.n; ++i) bc_apply(t.ops[c.op[i]], g, R, out);
  }
};

}  // namespace

extern "C" {

// every entry from q into out, whose interior the caller has filled; returns the kept ones
int ghost_out(int nb, const int32_t* dims, int ncut, const int32_t* cuts, int nbc, const int32_t* bcs, const double* T_wall,
              const double* q_inf, double g, double R, int reverse, double* const* q, double* const* out) {
  const int64_t maxc[6] = {0, 0, 0, 0, 0, 0};
  const Table x(nb, dims, ncut, cuts, nbc, bcs, T_wall, q_inf, g, R, maxc, false);
  const int n = (int)x.t.entries.size();
  for (int r = 0; r < n; ++r) {
    const GhostEntry& e = x.t.entries[reverse ? n - 1 - r : r];
    double v5[5];
    x.value(q, e.sb, e.sc, e.chain, v5);
    for (int v = 0; v < 5; ++v) out[e.tb][v * x.N[e.tb] + e.tc] = v5[v];
  }
  return x.t.nkept;
}

// the first launch in place on q, its records among its entries, into
// snap[face]; returns the late entries
int ghost_snaps(int nb, const int32_t* dims, int ncut, const int32_t* cuts, int nbc, const int32_t* bcs,
                const double* T_wall, const double* q_inf, double g, double R, int reverse, double* const* q,
                const int64_t* maxcells, double* const* snap) {
  int64_t maxc[6];
  for (int f = 0; f < 6; ++f) maxc[f] = maxcells[f];
  const Table x(nb, dims, ncut, cuts, nbc, bcs, T_wall, q_inf, g, R, maxc, true);
  const int n1 = x.t.ndirect + x.t.nstaged, n = n1 + (int)x.t.snaps.size();
  for (int r = 0; r < n; ++r) {
    const int i = reverse ? n - 1 - r : r;
    double v5[5];
    if (i < n1) {
      const GhostEntry& e = x.t.entries[i];
      x.value(q, e.sb, e.sc, e.chain, v5);
      if (i < x.t.ndirect)
        for (int v = 0; v < 5; ++v) q[e.tb][v * x.N[e.tb] + e.tc] = v5[v];
    } else {
      const GhostSnap& s = x.t.snaps[i - n1];
      x.value(q, s.sb, s.sc, s.chain, v5);
      for (int v = 0; v < 5; ++v) snap[s.face][s.off + v * s.stride] = v5[v];
    }
  }
  return x.t.nlate;
}

}

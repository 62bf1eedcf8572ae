// Test-only host build of the inviscid RHS kernel's slot maps (CrossGeom in
// famrdp-jax_amd/csrc/famrdp_tiles.h): every slot holds one cell, and every
// cell a face reads has the slot that step() names.  Compiled with
// --cuda-host-only; never loaded by the product.
#include <cstdint>

#include "famrdp_tiles.h"

using namespace famrdp;

namespace {

template <int TI, int TJ, int TK>
int64_t check() {
  using C = CrossGeom<TI, TJ, TK>;
  using W = WideGeom<TI, TJ, TK>;
  int64_t bad = 0;
  const int ext[3] = {TI, TJ, TK};
  for (int h = 0; h < C::NC; ++h) {
    const Loc3 l = C::cell(h);
    const int c[3] = {l.x, l.y, l.z};
    int out = 0;
    for (int e = 0; e < 3; ++e) {
      if (c[e] < -2 || c[e] > ext[e] + 1) ++bad;
      out += c[e] < 0 || c[e] >= ext[e];
    }
    if (out > 1 || (out == 0) != (h < C::NT)) ++bad;
    for (int g = 0; g < h; ++g) {
      const Loc3 o = C::cell(g);
      if (o.x == l.x && o.y == l.y && o.z == l.z) ++bad;
    }
  }
  for (int h = 0; h < C::NF; ++h) {
    const int D = W::face_axis_of(h);
    const Loc3 l = W::face_cell(h);
    for (int s = -2; s <= 1; ++s) {
      const int got = C::step(l, D, s);
      if (got < 0 || got >= C::NC) { ++bad; continue; }
      const Loc3 n = C::cell(got);
      if (n.x != l.x + (D == 0 ? s : 0) || n.y != l.y + (D == 1 ? s : 0) || n.z != l.z + (D == 2 ? s : 0)) ++bad;
    }
  }
  if (C::NTH < C::NF || C::NTH > 1024) ++bad;
  return bad;
}

}  // namespace

extern "C" int64_t cross_bad(int ti, int tj, int tk) {
  if (ti == 4 && tj == 4 && tk == 4) return check<4, 4, 4>();
  if (ti == 3 && tj == 4 && tk == 5) return check<3, 4, 5>();   // no two extents alike
  return -1;
}

// Test-only host build of the wide stage kernel's slot maps (WideGeom in
// famrdp-jax_amd/csrc/famrdp_tiles.h): every slot names one cell or face, the
// step maps reach the slot of the neighbour they are read for, and the faces
// of a tile cell are the slots of its neighbours' faces.  Compiled with
// --cuda-host-only; never loaded by the product.
#include <cstdint>

#include "famrdp_tiles.h"

using namespace famrdp;

namespace {

bool same(Loc3 a, Loc3 b) { return a.x == b.x && a.y == b.y && a.z == b.z; }
Loc3 step(Loc3 l, int e, int s) { return Loc3{l.x + (e == 0 ? s : 0), l.y + (e == 1 ? s : 0), l.z + (e == 2 ? s : 0)}; }

// FACES: the kernel has a thread per face as well
template <int TI, int TJ, int TK, bool FACES = true>
int64_t check() {
  using T = FusedGeom<TI, TJ, TK>;
  using W = WideGeom<TI, TJ, TK>;
  int64_t bad = 0;
  for (int h = 0; h < T::NPV; ++h)
    if (!same(W::pv_cell(h), T::pv_cell(h)) || T::pv_slot(W::pv_cell(h).x, W::pv_cell(h).y, W::pv_cell(h).z) != h) ++bad;
  for (int h = 0; h < T::NG; ++h) {
    const Loc3 l = W::g_cell(h);
    if (!same(l, T::g_cell(h))) ++bad;
    for (int e = 0; e < 3; ++e)
      for (int s = -1; s <= 1; s += 2) {   // the tensor's differences
        const Loc3 n = step(l, e, s);
        const int got = W::pv_step(l, e, s);
        if (got < 0 || got >= T::NPV || !same(T::pv_cell(got), n)) ++bad;
        if (h >= T::NT) continue;          // the divergence of a tile cell
        const int g = W::g_step(l, e, s);
        if (g < 0 || g >= T::NG || !same(T::g_cell(g), n)) ++bad;
      }
  }
  int64_t faces[3] = {0, 0, 0};
  for (int h = 0; h < W::NF; ++h) {
    const int D = W::face_axis_of(h);
    const Loc3 l = W::face_cell(h);
    ++faces[D];
    const int c[3] = {l.x, l.y, l.z}, ext[3] = {TI, TJ, TK};
    for (int e = 0; e < 3; ++e)
      if (c[e] < 0 || c[e] > ext[e] - (e == D ? 0 : 1)) ++bad;
    for (int s = -2; s <= 1; ++s) {
      const int got = W::pv_step(l, D, s);
      if (got < 0 || got >= T::NPV || !same(T::pv_cell(got), step(l, D, s))) ++bad;
    }
  }
  if (faces[0] != T::F0 || faces[1] != T::F1 || faces[2] != T::F2) ++bad;
  for (int h = 0; h < T::NT; ++h) {
    const Loc3 l = T::g_cell(h);
    const int lo[3] = {W::template low_face<0>(l.x, l.y, l.z), W::template low_face<1>(l.x, l.y, l.z),
                       W::template low_face<2>(l.x, l.y, l.z)};
    const int up[3] = {W::template high_face<0>(), W::template high_face<1>(), W::template high_face<2>()};
    for (int e = 0; e < 3; ++e) {
      if (lo[e] < 0 || lo[e] + up[e] >= W::NF) { ++bad; continue; }
      if (W::face_axis_of(lo[e]) != e || !same(W::face_cell(lo[e]), l)) ++bad;
      if (W::face_axis_of(lo[e] + up[e]) != e || !same(W::face_cell(lo[e] + up[e]), step(l, e, 1))) ++bad;
    }
  }
  if (W::NGW < T::NG || W::NTH - W::NGW < W::NF || W::NGW % 64 != 0 || (FACES ? W::NTH : W::NGW) > 1024) ++bad;
  return bad;
}

}  // namespace

extern "C" int64_t wide_bad(int ti, int tj, int tk) {
  if (ti == 3 && tj == 4 && tk == 4) return check<3, 4, 4>();
  if (ti == 4 && tj == 4 && tk == 8) return check<4, 4, 8>();
  if (ti == 4 && tj == 8 && tk == 8) return check<4, 8, 8, false>();   // the viscous RHS kernel's
  if (ti == 3 && tj == 4 && tk == 5) return check<3, 4, 5>();   // no two extents alike
  return -1;
}

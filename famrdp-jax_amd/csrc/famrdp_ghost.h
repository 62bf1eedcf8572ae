// Ghost cells of a step in one pass: the halo exchange (mesh/halo.py:56-92, all
// copies read the pre-exchange arrays, the final writer wins) followed by the
// boundary conditions (physics/bc/dispatch.py:11-32, faces in order, each on
// the result of the ones before).
//
// A ghost cell's final value is a chain of at most six boundary operations
// (one per face) on the pre-exchange value of one source cell, so the whole
// sequence -- two launches for the exchange and one per face with a boundary
// condition -- becomes a table of (target, source, chain), resolved once per
// plan by following the sequence cell by cell.  An entry whose source is
// nobody's target is applied directly; the few others (edges and corners) read
// their sources into a staging buffer in the first launch and are written in a
// second one, with the entries that overwrite such a source.  Without any, one
// launch does it all.  The table builder runs on the host and is checked there
// against the sequence itself.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "famrdp_kernels.h"

namespace famrdp {

// Target cell tc of block tb takes chain `chain` of source cell sc of block sb
// (sb < 0: the chain starts with a free stream and reads nothing).
struct GhostEntry {
  int32_t tb, tc, sb, sc, chain;
};
constexpr int GHOST_CHAIN = 6;
struct GhostChain {
  int32_t n, op[GHOST_CHAIN];   // indices into the table of BcEntry
};
// The same for a value that is only recorded (the reverse sweep linearises
// isothermal walls at it): variable v goes to snap[face][off + v * stride].
struct GhostSnap {
  int32_t sb, sc, chain, face;
  int64_t off, stride;
};

// One boundary operation on a cell's conservative variables (physics/bc/
// wall.py:7-64, symmetry.py:8-11, farfield.py:7-21).
FD void bc_apply(const BcEntry& e, double gamma, double R, double q[5]) {
  switch (e.kind) {
    case BC_WALL_ADIABATIC:
      q[1] = -q[1]; q[2] = -q[2]; q[3] = -q[3];
      break;
    case BC_WALL_ISOTHERMAL: {   // bc/wall.py:35-58
      const double rho_i = q[0];
      const double ke_i = 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / rho_i;
      const double p_g = (gamma - 1.0) * (q[4] - ke_i);
      const double rho_g = p_g / (R * e.T_wall);
      const double scale = rho_g / rho_i;
      const double mu = -q[1] * scale, mv = -q[2] * scale, mw = -q[3] * scale;
      const double ke_g = 0.5 * (mu * mu + mv * mv + mw * mw) / rho_g;
      q[0] = rho_g; q[1] = mu; q[2] = mv; q[3] = mw; q[4] = p_g / (gamma - 1.0) + ke_g;
      break;
    }
    case BC_MIRROR_NORMAL: {
      const int ax = e.face / 2;
      q[1] = ax == 0 ? -q[1] : q[1];
      q[2] = ax == 1 ? -q[2] : q[2];
      q[3] = ax == 2 ? -q[3] : q[3];
      break;
    }
    case BC_FARFIELD:
      for (int v = 0; v < 5; ++v) q[v] = e.q_inf[v];
      break;
    default:  // BC_EXTRAPOLATE: the source's value
      break;
  }
}

// mirror pairs of a face (bc/base.py:21-33); extrapolation reads the first
// interior layer
FD void bc_pair(const BcEntry& e, int ghost, int n, int gl, int& outer, int& inner) {
  const bool lo = (e.face % 2) == 0;
  outer = lo ? gl : n - 1 - gl;
  inner = lo ? 2 * ghost - 1 - gl : n - 2 * ghost + gl;
  if (e.kind == BC_EXTRAPOLATE) inner = lo ? ghost : n - 1 - ghost;
}

// Ghost cells of a block, numbered: the i slabs, then the j slabs of the
// remaining planes, then the k slabs of the remaining rows.
struct GhostShell {
  int g, n[3];
  int64_t b1, b2, size;
  GhostShell(int ghost, const int32_t* d) : g(ghost), n{d[0], d[1], d[2]} {
    const int64_t mi = n[0] - 2 * g, mj = n[1] - 2 * g;
    b1 = (int64_t)2 * g * n[1] * n[2];
    b2 = b1 + mi * 2 * g * n[2];
    size = b2 + mi * mj * 2 * g;
  }
  static int layer(int x, int n, int g) { return x < g ? x : (x >= n - g ? x - (n - 2 * g) : -1); }
  // number of the ghost cell (i, j, k), or -1 for an interior cell
  int64_t index(int i, int j, int k) const {
    const int li = layer(i, n[0], g);
    if (li >= 0) return ((int64_t)li * n[1] + j) * n[2] + k;
    const int lj = layer(j, n[1], g);
    if (lj >= 0) return b1 + ((int64_t)(i - g) * 2 * g + lj) * n[2] + k;
    const int lk = layer(k, n[2], g);
    if (lk >= 0) return b2 + ((int64_t)(i - g) * (n[1] - 2 * g) + (j - g)) * 2 * g + lk;
    return -1;
  }
  int64_t index_of(int32_t cell) const {
    const int k = cell % n[2], r = cell / n[2];
    return index(r / n[1], r % n[1], k);
  }
  // calls f(cell, number) for every ghost cell, cells ascending
  template <class F>
  void each(F f) const {
    for (int i = 0; i < n[0]; ++i)
      for (int j = 0; j < n[1]; ++j) {
        const bool whole = layer(i, n[0], g) >= 0 || layer(j, n[1], g) >= 0;
        const int32_t row = (int32_t)(((int64_t)i * n[1] + j) * n[2]);
        int64_t s = index(i, j, 0);           // numbers run along a row
        for (int k = 0; k < n[2]; ++k) {
          if (!whole && k == g && n[2] > 2 * g) k = n[2] - g;
          f(row + k, s++);
        }
      }
  }
};

// The ghost table of a plan: copy() takes the copies of the exchange, then
// boundary() the boundary conditions -- bc[f] those of face f (at most one per
// block), in the order of the blocks' application -- and finish() orders the
// entries.
struct GhostTable {
  struct Val {
    int32_t sb, sc, chain;   // chain -1: untouched
    int32_t ss;              // the source's number in its block's shell, -1 for an interior cell
  };
  int ghost;
  std::vector<GhostShell> shell;
  std::vector<std::vector<Val>> val;       // per block and ghost cell
  std::vector<BcEntry> ops;
  std::vector<GhostChain> chains;          // 0: the value itself
  // [direct | staged | late direct | kept]: kept are the ghost cells that
  // nothing writes, as copies of themselves, for a step into other arrays
  std::vector<GhostEntry> entries;
  int ndirect = 0, nstaged = 0, nlate = 0, nkept = 0;
  std::vector<GhostSnap> snaps;
  std::vector<int32_t> snap_ss;            // Val::ss of the recorded values

  GhostTable(int ghost_, int nblocks, const int32_t* dims) : ghost(ghost_) {
    chains.push_back(GhostChain{0, {0, 0, 0, 0, 0, 0}});
    for (int b = 0; b < nblocks; ++b) {
      shell.emplace_back(ghost, dims + 3 * b);
      val.emplace_back((size_t)shell[b].size, Val{0, 0, -1, -1});
    }
  }

  // the exchange's copy of cell sc of block sb to the ghost cell (i, j, k) of
  // block tb; a later copy wins
  void copy(int tb, int i, int j, int k, int sb, int32_t sc) {
    val[tb][(size_t)shell[tb].index(i, j, k)] = Val{sb, sc, 0, (int32_t)shell[sb].index_of(sc)};
  }

  // The exchange's final copies, ordered by target.
  void halo(std::vector<HaloEntry>& out) const {
    size_t n = 0;
    for (const auto& vals : val)
      for (const Val& v : vals) n += v.chain >= 0;
    out.reserve(n);
    for (int b = 0; b < (int)shell.size(); ++b)
      shell[b].each([&](int32_t c, int64_t s) {
        const Val& v = val[b][(size_t)s];
        if (v.chain >= 0) out.push_back(HaloEntry{b, c, v.sb, v.sc});
      });
  }

  // The boundary conditions, in order; with `snap`, the inner layers of
  // isothermal faces as they are when the face is applied.
  void boundary(const std::vector<BcEntry> (&bc)[6], const int64_t (&maxcells)[6], bool snap) {
    size_t nsnap = 0;
    for (int f = 0; f < 6; ++f)
      for (const BcEntry& op : bc[f])
        if (snap && op.kind == BC_WALL_ISOTHERMAL) nsnap += (size_t)(ghost * maxcells[f]);
    snaps.reserve(nsnap);
    snap_ss.reserve(nsnap);
    std::vector<int32_t> longer;   // chain -> that chain and the operation at hand, -1: not made yet
    for (int f = 0; f < 6; ++f) {
      const int ax = f / 2, t1 = ax == 0 ? 1 : 0, t2 = ax == 2 ? 1 : 2;
      for (size_t e = 0; e < bc[f].size(); ++e) {
        const BcEntry& op = bc[f][e];
        const int32_t iop = (int32_t)ops.size();
        ops.push_back(op);
        longer.assign(chains.size(), -1);
        const GhostShell& sh = shell[op.block];
        auto& vals = val[op.block];
        int x[3];
        for (x[t1] = 0; x[t1] < sh.n[t1]; ++x[t1])
          for (x[t2] = 0; x[t2] < sh.n[t2]; ++x[t2])
            for (int gl = 0; gl < ghost; ++gl) {
              int outer, inner;
              bc_pair(op, ghost, sh.n[ax], gl, outer, inner);
              x[ax] = inner;
              const int32_t ci = (int32_t)(((int64_t)x[0] * sh.n[1] + x[1]) * sh.n[2] + x[2]);
              const int64_t si = sh.index(x[0], x[1], x[2]);
              Val v = si >= 0 && vals[(size_t)si].chain >= 0 ? vals[(size_t)si] : Val{op.block, ci, 0, (int32_t)si};
              if (snap && op.kind == BC_WALL_ISOTHERMAL) {
                snap_ss.push_back(v.ss);
                snaps.push_back(GhostSnap{v.sb, v.sc, v.chain, f,
                                          ((int64_t)e * ghost + gl) * 5 * maxcells[f] + (int64_t)x[t1] * sh.n[t2] + x[t2],
                                          maxcells[f]});
              }
              if (op.kind == BC_FARFIELD) v = Val{-1, 0, 0, -1};
              if (op.kind != BC_EXTRAPOLATE) {
                // (a cell read here is never one this operation has written: longer covers its chain)
                int32_t& next = longer[(size_t)v.chain];
                if (next < 0) {
                  GhostChain c = chains[(size_t)v.chain];
                  c.op[c.n++] = iop;
                  next = (int32_t)chains.size();
                  chains.push_back(c);
                }
                v.chain = next;
              }
              x[ax] = outer;
              vals[(size_t)sh.index(x[0], x[1], x[2])] = v;
            }
      }
    }
  }

  // Entries in launch order.
  void finish() {
    // per target: 1 a staged entry or a snapshot reads its old value, 2 it is staged itself
    std::vector<std::vector<char>> flag(shell.size());
    for (size_t b = 0; b < shell.size(); ++b) flag[b].assign((size_t)shell[b].size, 0);
    auto waits = [&](int32_t sb, int32_t ss) { return sb >= 0 && ss >= 0 && val[(size_t)sb][(size_t)ss].chain >= 0; };
    for (size_t i = 0; i < snaps.size(); ++i)
      if (waits(snaps[i].sb, snap_ss[i])) flag[(size_t)snaps[i].sb][(size_t)snap_ss[i]] |= 1;
    int64_t total = 0;
    nstaged = nlate = nkept = 0;
    for (size_t b = 0; b < val.size(); ++b)
      for (size_t s = 0; s < val[b].size(); ++s) {
        const Val& v = val[b][s];
        if (v.chain < 0) { ++nkept; continue; }
        ++total;
        if (!waits(v.sb, v.ss)) continue;
        flag[(size_t)v.sb][(size_t)v.ss] |= 1;
        flag[b][s] |= 2;
        ++nstaged;
      }
    for (size_t b = 0; b < val.size(); ++b)
      for (size_t s = 0; s < val[b].size(); ++s) nlate += flag[b][s] == 1 && val[b][s].chain >= 0;
    ndirect = (int)(total - nstaged - nlate);
    entries.resize((size_t)total + nkept);
    GhostEntry *direct = entries.data(), *staged = direct + ndirect, *late = staged + nstaged, *kept = late + nlate;
    for (int b = 0; b < (int)shell.size(); ++b)
      shell[b].each([&](int32_t c, int64_t s) {
        const Val& v = val[b][(size_t)s];
        if (v.chain < 0) { *kept++ = GhostEntry{b, c, b, c, 0}; return; }
        const int f = flag[b][(size_t)s];
        GhostEntry*& to = f >= 2 ? staged : (f == 1 ? late : direct);
        *to++ = GhostEntry{b, c, v.sb, v.sc, v.chain};
      });
  }
};

}  // namespace famrdp

// Reverse-mode stage kernels of the TVD-RK3 step.
//
// One RK stage  q_out = a q0 + b (q_s + dt L(q_s))  is reversed by two kernels
// (no atomics, deterministic).  Every cell's reverse needs, along each axis,
// the cotangents of four faces and of three limited slopes; instead of passing
// them through memory, each axis is swept so that they stay with the wave.  A
// wave never waits for another one: no barriers, LDS only as the threads' own
// store.  Thirteen doubles per cell go from the first kernel to the second:
//   k_vjp_i   two independent sweeps along i, k-neighbours in the wave's lanes:
//             sweep_visc  the cotangent of the viscous flux tensor G from the
//                         divergence at the six neighbours, the reverse of G
//                         into d/d(u, v, w, T) and d/d(central differences),
//                         and of the latter the i and k ones; the j ones are
//                         passed on;
//             sweep_ik    the inviscid i and k axes;
//   k_vjp_j   the j axis: a wave holds 64 columns (i, k) and marches along j; a
//             cell's axes complete, it adds the viscous part, maps the
//             primitive cotangent to conservative variables and applies the RK
//             coefficients.
// Functions cite the forward code they reverse in famrdp_jax (rhs/invscd.py,
// rhs/viscous.py, solver/step.py).  This file is its own translation unit,
// compiled with the default machine scheduler (the rest of the library uses
// the max-ilp one, with which the two inviscid sweeps spill or come close).
//
// One stage of 10^6 cells (curvilinear 96^3) takes 142 + 88 us (133 + 87 with
// reciprocal roots from seeds, whose squares round twice); two gather
// kernels that passed 46 doubles per cell (three faces' state cotangents, the
// viscous ones) took 223 + 184 us.  What bounds them now: k_vjp_j moves 42
// doubles a cell that no other access could save (68 us at the 4.9 TB/s of a
// large copy); k_vjp_i 48 (78 us), at two waves per SIMD whose loads and FP64
// chains overlap only with each other's.  Its two sweeps as launches of their
// own: 73 + 75 us.  Measured and not kept: the next step's loads issued a step
// ahead (the face's reverse alone takes 156 registers: spills, 101 us for
// sweep_ik); sweep_visc at three waves per SIMD (164 registers with its carried
// values in LDS: 74 us, and longer waits for small blocks).
#include "famrdp_kernels.h"
#include "famrdp_adjoint.h"
#include "famrdp_reverse.h"

namespace famrdp {

// Cells are addressed with 32-bit element indices (an adjoint plan's blocks
// hold fewer than 2^29 cells: famrdp_plan_create refuses larger ones), loads
// and stores through a 32-bit byte offset from a base that is the same for the whole wave -- the base stays in scalar
// registers and a cell costs one 32-bit offset, however many arrays it reads
// (global loads and stores: the pointers come from the device block table).
__device__ __forceinline__ double rd(const double* __restrict__ a, unsigned i) {
  return *(gmem_cdouble*)(reinterpret_cast<const char*>(a) + (i << 3));
}
__device__ __forceinline__ gmem_double& at(double* a, unsigned i) {
  return *(gmem_double*)(reinterpret_cast<char*>(a) + (i << 3));
}

__device__ __forceinline__ void rd_prim(const double* __restrict__ q, int64_t N, unsigned c, double g, double pv[5]) {
  double qc[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) qc[v] = rd(q + v * N, c);
  cons_to_prim_fast(qc, g, pv);
}

// ---------------------------------------------------------------------------
// one axis of the inviscid part, swept (rhs/invscd.py:53-131 reversed)
// ---------------------------------------------------------------------------

// What a sweep along an axis carries when it processes cell s, s increasing.
// The registers of the face's reverse decide how much a wave can hold besides,
// so only what the face needs as it is stays in registers: the primitives of
// cell s and the left state of the face (s-1 | s).  The rest lies in the
// thread's own LDS column: primitives, scaled cotangent and axis metrics of
// cell s-1, the difference p(s-1) - p(s-2), the cotangent of the right state
// of face (s-2 | s-1), what cell s-1 already holds (the slope of s-2 reaching
// up, and what the caller adds) and the incomplete sum of cell s-2.
struct AxisSweep {
  double pc[5], pLn[5];
  double* rest;
};
enum : int { SW_PM = 0, SW_DA = 5, SW_LPR = 10, SW_CARRY = 15, SW_ACC = 20, SW_MR = 25, SW_KD = 30, SW_N = 33 };
constexpr int SWEEP_NT = 256;
__device__ __forceinline__ double& sw(const AxisSweep& st, int i) { return st.rest[i * SWEEP_NT]; }
// x is computed by here (not later, from operands that would stay alive)
__device__ __forceinline__ void pin(double (&x)[5]) {
#pragma unroll
  for (int v = 0; v < 5; ++v) asm volatile("" : "+v"(x[v]));
}

// What one step of a sweep reads: the state of the cell after (s+1), the
// cotangent, volume and metrics of cell s.
template <int NK>
struct SweepLoads {
  double q[5], l[5], vol, k[NK];
};
// k rows from row k0, and (NK = 6) from row 6
template <int NK>
__device__ __forceinline__ void sweep_load(SweepLoads<NK>& x, const BlockDesc& b, const double* __restrict__ qs,
                                           const double* __restrict__ lin, unsigned c, unsigned cn, int k0) {
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    x.l[v] = rd(lin + v * b.N, c);
    x.q[v] = rd(qs + v * b.N, cn);
  }
  x.vol = rd(b.vol, c);
#pragma unroll
  for (int m = 0; m < 3; ++m) x.k[m] = rd(b.kxyz + (k0 + m) * b.N, c);
  if constexpr (NK == 6) {
#pragma unroll
    for (int m = 0; m < 3; ++m) x.k[3 + m] = rd(b.kxyz + (6 + m) * b.N, c);
  }
}

// The cotangent of a cell's flux difference, per unit of twice the flux:
// c_mu lin / (2 (vol + 1e-300)); a face takes it from the cell on its right
// and, negated, from the cell on its left, where those cells difference it.
//
// One step: cell s with primitives st.pc, pn = p(s+1), mr and kd of cell s.
// vl, vr: cells s-1 and s difference their faces (2 .. n-3); face: the face
// (s-1 | s) exists (left cell in 1 .. n-3); in: cell s-1 has a slope (1 ..
// n-2); kp: added to what cell s holds.  Completes cell s-2 into out; st then
// stands at s+1.
template <int LIM>
__device__ __forceinline__ void axis_step(AxisSweep& st, const double pn[5], const double mr[5], const double kd[3],
                                          bool vl, bool vr, bool face, bool in, double cg2, double gm1h,
                                          const double kp[5], double out[5]) {
  double pLs[5], lpl[5] = {0, 0, 0, 0, 0}, lpr[5] = {0, 0, 0, 0, 0};
  {
    double pm[5], pRs[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) pm[v] = sw(st, SW_PM + v);
    muscl_cell<LIM>(pm, st.pc, pn, pLs, pRs);
    if (face) {
      double f[5], S[3];
#pragma unroll
      for (int m = 0; m < 3; ++m) S[m] = 0.5 * (sw(st, SW_KD + m) + kd[m]);
#pragma unroll
      for (int v = 0; v < 5; ++v) f[v] = (vr ? mr[v] : 0.0) - (vl ? sw(st, SW_MR + v) : 0.0);
      roe_flux2_vjp(st.pLn, pRs, S, cg2, gm1h, f, lpl, lpr);
    }
  }
  pin(lpl);
  pin(lpr);
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double B = st.pc[v] - sw(st, SW_PM + v), lp = sw(st, SW_LPR + v);
    double lA = 0.0, lB = 0.0;
    if (in) limiter_vjp_t<LIM>(sw(st, SW_DA + v), B, 0.5 * (lpl[v] - lp), lA, lB);
    out[v] = sw(st, SW_ACC + v) - lA;
    sw(st, SW_ACC + v) = ((lp + lpl[v]) + (lA - lB)) + sw(st, SW_CARRY + v);
    sw(st, SW_CARRY + v) = lB + kp[v];
    sw(st, SW_DA + v) = B;
    sw(st, SW_LPR + v) = lpr[v];
    sw(st, SW_PM + v) = st.pc[v];
    sw(st, SW_MR + v) = mr[v];
    st.pc[v] = pn[v];
    st.pLn[v] = pLs[v];
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) sw(st, SW_KD + m) = kd[m];
}

// Start of a sweep whose first step processes cell s: c3, c2, c1 the cells
// s-2, s-1 and s.
template <int LIM>
__device__ __forceinline__ void sweep_begin(AxisSweep& st, const BlockDesc& b, const double* __restrict__ qs,
                                            const double* __restrict__ lin, unsigned c3, unsigned c2, unsigned c1,
                                            int k0, double g, double hcm) {
  double p0[5], pm[5], pr[5];
  rd_prim(qs, b.N, c3, g, p0);
  rd_prim(qs, b.N, c2, g, pm);
  rd_prim(qs, b.N, c1, g, st.pc);
  muscl_cell<LIM>(p0, pm, st.pc, st.pLn, pr);
  const double r = hcm * rcp_hd(rd(b.vol, c2) + 1e-300);
#pragma unroll
  for (int v = 0; v < SW_N; ++v) sw(st, v) = 0.0;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    sw(st, SW_PM + v) = pm[v];
    sw(st, SW_MR + v) = r * rd(lin + v * b.N, c2);
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) sw(st, SW_KD + m) = rd(b.kxyz + (k0 + m) * b.N, c2);
}

// x of the lane below / above (the end lane of the wave keeps its own): a
// wave-wide DPP shift, two moves for a double and no LDS
template <int CTRL>
__device__ __forceinline__ double lane_shift(double x) {
  typedef int pair2 __attribute__((__vector_size__(8)));
  pair2 u = __builtin_bit_cast(pair2, x);
  u[0] = __builtin_amdgcn_update_dpp(u[0], u[0], CTRL, 0xf, 0xf, false);
  u[1] = __builtin_amdgcn_update_dpp(u[1], u[1], CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, u);
}
__device__ __forceinline__ double lane_below(double x) { return lane_shift<0x138>(x); }   // wave_shr:1
__device__ __forceinline__ double lane_above(double x) { return lane_shift<0x130>(x); }   // wave_shl:1

// The k axis of the 64 consecutive cells of one plane a wave holds: each lane
// its cell's low face, the rest from the lanes beside it.  A lane's result
// needs three lanes either side, so lanes 3 .. 60 are complete.  Rows end
// inside a wave: faces and slopes exist by the cell's own k, and what a lane
// takes from the next row is a face or slope that does not exist there (zero).
template <int LIM>
__device__ __forceinline__ void lanes_k(const double pv[5], const double mr[5], const double kd[3], int k, int nk,
                                        double cg2, double gm1h, double out[5]) {
  double pL[5], pR[5], dA[5], dB[5], f[5], lpl[5] = {0, 0, 0, 0, 0}, lpr[5] = {0, 0, 0, 0, 0};
  double S[3];
  {
    double pb[5], pa[5], ph[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      pb[v] = lane_below(pv[v]);
      pa[v] = lane_above(pv[v]);
      dA[v] = pv[v] - pb[v];
      dB[v] = pa[v] - pv[v];
    }
    muscl_cell<LIM>(pb, pv, pa, ph, pR);
    const bool vl = k - 1 >= 2 && k - 1 <= nk - 3, vr = k >= 2 && k <= nk - 3;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      pL[v] = lane_below(ph[v]);
      const double mb = lane_below(mr[v]);
      f[v] = (vr ? mr[v] : 0.0) - (vl ? mb : 0.0);
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) S[m] = 0.5 * (lane_below(kd[m]) + kd[m]);
  }
  if (k >= 2 && k <= nk - 2) roe_flux2_vjp(pL, pR, S, cg2, gm1h, f, lpl, lpr);
  const bool in = k >= 1 && k <= nk - 2;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double lh = lane_above(lpl[v]);      // left state of the cell's high face
    double lA = 0.0, lB = 0.0;
    if (in) limiter_vjp_t<LIM>(dA[v], dB[v], 0.5 * (lh - lpr[v]), lA, lB);
    out[v] = ((lpr[v] + lh) + (lA - lB)) + (lane_below(lB) - lane_above(lA));
  }
}

// ---------------------------------------------------------------------------
// viscous part (rhs/viscous.py:86-108 and 30-84 reversed)
// ---------------------------------------------------------------------------

// What the viscous reverse needs of a cell besides its place: u, v, w, T and
// the momentum and energy cotangents (unscaled: every result is linear in
// them and takes c_mu at the end).
struct ViscCell {
  double w[4], m[4];
};
__device__ __forceinline__ void load_visc(const double* __restrict__ qs, const double* __restrict__ lin, int64_t N,
                                          unsigned c, const Gas& gas, ViscCell& x) {
  double pv[5];
  rd_prim(qs, N, c, gas.gamma, pv);
  x.w[0] = pv[1];
  x.w[1] = pv[2];
  x.w[2] = pv[3];
  x.w[3] = temperature_fast(pv, gas.R);
#pragma unroll
  for (int r = 0; r < 4; ++r) x.m[r] = rd(lin + (r + 1) * N, c);
}

// lG += sgn / 2 x (kxyz[l, :] times the cotangents of a neighbour): the
// divergence at x - e_l holds +G(x) / 2, at x + e_l it holds -G(x) / 2.
// kh = kxyz[l, :] / 2 of the neighbour.
__device__ __forceinline__ void add_lG(double lG[9], const double m[4], const double kh[3], double sgn) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int jj = 0; jj < 3; ++jj) lG[gidx(r, jj)] += (sgn * kh[jj]) * m[r];
}

// ---------------------------------------------------------------------------
// a cell whose axes are summed (lpv, cotangent of its primitives): viscous
// gather, primitive -> conservative, RK coefficients
//   stage 3: lout = 2/3 lin + g                      (its share of l0, lin / 3,
//            waits: lin is l0 itself, still read by other waves)
//   stage 2: l0 = l0 / 3 + 3/4 lin, lout = 1/4 lin + g
//   stage 1: l0 += lin + g
// ---------------------------------------------------------------------------
__device__ __forceinline__ void cell_vjp_finish(const BlockDesc& b, const double* __restrict__ qs, const double* lin,
                                                double* lout, int j, unsigned y, const Gas& gas, int stage,
                                                double lpv[5]) {
  const int64_t N = b.N;
  double q[5], pv[5], ls4[4];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    q[v] = rd(qs + v * N, y);
    lpv[v] += rd(b.fs + v * N, y);
  }
  cons_to_prim_fast(q, gas.gamma, pv);
  // viscous: vs holds what sweep_visc summed (u, v, w, T) and the cotangents
  // of the cell's central differences along j
  const unsigned jm = y + (unsigned)((wrap_m(j, b.nj) - j) * b.nk), jp = y + (unsigned)((wrap_p(j, b.nj) - j) * b.nk);
#pragma unroll
  for (int s = 0; s < 4; ++s)
    ls4[s] = rd(b.vs + s * N, y) + 0.5 * (rd(b.vs + (4 + s) * N, jm) - rd(b.vs + (4 + s) * N, jp));
  lpv[1] += ls4[0]; lpv[2] += ls4[1]; lpv[3] += ls4[2];
  temperature_vjp(pv, gas.R, ls4[3], lpv[0], lpv[4]);
  double gq[5] = {0, 0, 0, 0, 0};
  cons_to_prim_vjp(q, gas.gamma, lpv, gq);
  // ---- RK coefficients (solver/step.py:45-53 reversed)
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double li = rd(lin + v * N, y);
    gmem_double& l0 = at(b.l0 + v * N, y);
    if (stage == 3) {
      at(lout + v * N, y) = (2.0 / 3.0) * li + gq[v];
    } else if (stage == 2) {
      l0 = (1.0 / 3.0) * l0 + 0.75 * li;
      at(lout + v * N, y) = 0.25 * li + gq[v];
    } else {
      l0 += li + gq[v];
    }
  }
}

// Stage selector for the reverse sweep: which buffers a stage reads/writes.
//   stage 3: qs = q2, lin = l0 (the cotangent of q_new), lout = lb
//   stage 2: qs = q1, lin = lb, lout = la
//   stage 1: qs = qh, lin = la
__device__ __forceinline__ void vjp_bufs(const BlockDesc& b, int stage, const double*& qs, const double*& lin,
                                         double*& lout) {
  qs = stage == 3 ? b.q2 : (stage == 2 ? b.q1 : b.qh);
  lin = stage == 3 ? b.l0 : (stage == 2 ? b.lb : b.la);
  lout = stage == 3 ? b.lb : (stage == 2 ? b.la : nullptr);
}

__device__ __forceinline__ double stage_cmu(int stage, double dt) {
  return stage == 3 ? (2.0 / 3.0) * dt : (stage == 2 ? 0.25 * dt : dt);
}

// The viscous part: a wave marches along i over 64 cells of a plane, lanes
// 2 .. 61 complete (a cell takes the difference cotangents of its neighbours,
// which take the state of theirs).  The rows of a plane are laid out with two
// cells of periodic image at either end (nk + 4 lanes a row), so the lanes
// beside a lane are its k-neighbours in the roll's sense too; planes and rows
// wrap in their index.  Step s reverses G at plane s -- i-neighbours carried,
// k-neighbours from the lanes, j-neighbours loaded -- and completes plane s-1.
__device__ __forceinline__ void sweep_visc(const BlockDesc& b, const SweepTile& tl, int stage, const Gas& gas,
                                           double dt) {
  const int lane = threadIdx.x & 63, ni = b.ni, nj = b.nj, nk = b.nk, ne = nj * (nk + 4);
  const int64_t N = b.N;
  const unsigned njk = (unsigned)nj * (unsigned)nk;
  const double *qs, *lin;
  double* lout;
  vjp_bufs(b, stage, qs, lin, lout);
  const double cmu = stage_cmu(stage, dt * b.dt_scale);
  const int e0 = tl.base - 2 + lane, e = e0 < 0 ? 0 : (e0 >= ne ? ne - 1 : e0);
  const int j = e / (nk + 4), ke = e % (nk + 4) - 2;
  const int k = ke < 0 ? ke + nk : (ke >= nk ? ke - nk : ke);
  const bool own = lane >= 2 && lane <= 61 && e0 < ne && ke >= 0 && ke < nk;
  const unsigned cp = (unsigned)(j * nk + k);
  const unsigned ojm = (unsigned)((wrap_m(j, nj) - j) * nk), ojp = (unsigned)((wrap_p(j, nj) - j) * nk);
  auto cell = [&](int s) -> unsigned { return (unsigned)(s < 0 ? s + ni : (s >= ni ? s - ni : s)) * njk + cp; };

  // planes s-1 and s: state, cotangents, kxyz[0, :] / 2
  ViscCell xm, xc;
  double km[3], kc[3];
  load_visc(qs, lin, N, cell(tl.p0 - 2), gas, xm);
  load_visc(qs, lin, N, cell(tl.p0 - 1), gas, xc);
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    km[m] = 0.5 * rd(b.kxyz + m * N, cell(tl.p0 - 2));
    kc[m] = 0.5 * rd(b.kxyz + m * N, cell(tl.p0 - 1));
  }
  double acc[4] = {0, 0, 0, 0};    // plane s-1 without the share of plane s
  double ldi[4] = {0, 0, 0, 0};    // cotangents of the i differences of plane s-1, halved
  for (int s = tl.p0 - 1; s <= tl.p1; ++s) {
    const unsigned c = cell(s), cn = cell(s + 1);
    ViscCell xn, xj;
    double kn[3], kk[9], lG[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, d[3][4], kj[3];
    load_visc(qs, lin, N, cn, gas, xn);
#pragma unroll
    for (int m = 0; m < 3; ++m) kn[m] = 0.5 * rd(b.kxyz + m * N, cn);
#pragma unroll
    for (int m = 3; m < 9; ++m) kk[m] = rd(b.kxyz + m * N, c);
#pragma unroll
    for (int m = 0; m < 3; ++m) kk[m] = 2.0 * kc[m];
    // j-neighbours
    load_visc(qs, lin, N, c + ojm, gas, xj);
#pragma unroll
    for (int m = 0; m < 3; ++m) kj[m] = 0.5 * rd(b.kxyz + (3 + m) * N, c + ojm);
    add_lG(lG, xj.m, kj, 1.0);
#pragma unroll
    for (int q = 0; q < 4; ++q) d[1][q] = -xj.w[q];
    load_visc(qs, lin, N, c + ojp, gas, xj);
#pragma unroll
    for (int m = 0; m < 3; ++m) kj[m] = 0.5 * rd(b.kxyz + (3 + m) * N, c + ojp);
    add_lG(lG, xj.m, kj, -1.0);
#pragma unroll
    for (int q = 0; q < 4; ++q) d[1][q] = 0.5 * (d[1][q] + xj.w[q]);
    // k-neighbours
    {
      double mb[4], ma[4], kb[3], ka[3];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        mb[q] = lane_below(xc.m[q]);
        ma[q] = lane_above(xc.m[q]);
        d[2][q] = 0.5 * (lane_above(xc.w[q]) - lane_below(xc.w[q]));
      }
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        const double h = 0.5 * kk[6 + m];
        kb[m] = lane_below(h);
        ka[m] = lane_above(h);
      }
      add_lG(lG, mb, kb, 1.0);
      add_lG(lG, ma, ka, -1.0);
    }
    // i-neighbours
    add_lG(lG, xm.m, km, 1.0);
    add_lG(lG, xn.m, kn, -1.0);
#pragma unroll
    for (int q = 0; q < 4; ++q) d[0][q] = 0.5 * (xn.w[q] - xm.w[q]);
    double l4[4] = {0, 0, 0, 0}, ld[3][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
    const double pv[5] = {0.0, xc.w[0], xc.w[1], xc.w[2], 0.0};
    viscous_flux_vjp(pv, xc.w[3], d, kk, gas.gamma, gas.R, b.mu0, gas.T0, gas.Ts, gas.Pr_lam, lG, l4[0], l4[1], l4[2],
                     l4[3], ld);
    const bool out1 = s > tl.p0 && own, out0 = s >= tl.p0 && s < tl.p1 && own;
    const unsigned cm = cell(s - 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (out1) at(b.vs + q * N, cm) = cmu * (acc[q] - 0.5 * ld[0][q]);
      if (out0) at(b.vs + (4 + q) * N, c) = cmu * ld[1][q];
      acc[q] = (l4[q] + ldi[q]) + 0.5 * (lane_below(ld[2][q]) - lane_above(ld[2][q]));
      ldi[q] = 0.5 * ld[0][q];
    }
    xm = xc;
    xc = xn;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      km[m] = kc[m];
      kc[m] = kn[m];
    }
  }
}

// The i and k axes: lanes 3 .. 60 hold the plane cells from base on, planes p0
// .. p1-1.  The wave starts three planes early and ends two late (the slopes
// and faces around its first and last plane).  Writes the sum of both axes
// (the cotangent of the five primitives) to fs.
template <int LIM>
__device__ __forceinline__ void sweep_ik(double* rest, const BlockDesc& b, const SweepTile& tl, int stage,
                                         const Gas& gas, double dt) {
  const int lane = threadIdx.x & 63, ni = b.ni, nk = b.nk;
  const int64_t N = b.N;
  const unsigned njk = (unsigned)b.nj * (unsigned)nk;
  const double *qs, *lin;
  double* lout;
  vjp_bufs(b, stage, qs, lin, lout);
  const double hcm = uniform(0.5 * stage_cmu(stage, dt * b.dt_scale));
  const double g = gas.gamma, cg2 = uniform(2.0 * g / (g - 1.0)), gm1h = uniform(0.5 * (g - 1.0));
  // the lane's plane cell (the nearest one where it lies outside the plane)
  const int cl = tl.base - 3 + lane;
  const unsigned cp = cl < 0 ? 0u : (cl >= (int)njk ? njk - 1u : (unsigned)cl);
  const int k = (int)(cp % (unsigned)nk);
  const bool own = lane >= 3 && lane <= 60 && cl < (int)njk;
  auto cell = [&](int s) -> unsigned { return (unsigned)(s < 0 ? 0 : (s >= ni ? ni - 1 : s)) * njk + cp; };

  AxisSweep st;
  st.rest = rest + threadIdx.x;
  sweep_begin<LIM>(st, b, qs, lin, cell(tl.p0 - 3), cell(tl.p0 - 2), cell(tl.p0 - 1), 0, g, hcm);
  SweepLoads<6> x;
  for (int s = tl.p0 - 1; s <= tl.p1 + 1; ++s) {
    double pn[5], mr[5], kd[3], out[5], kp[5] = {0, 0, 0, 0, 0};
    sweep_load(x, b, qs, lin, cell(s), cell(s + 1), 0);
    const double r = hcm * rcp_hd(x.vol + 1e-300);
#pragma unroll
    for (int v = 0; v < 5; ++v) mr[v] = r * x.l[v];
#pragma unroll
    for (int m = 0; m < 3; ++m) kd[m] = x.k[m];
    if (s >= tl.p0 && s < tl.p1) {
      lanes_k<LIM>(st.pc, mr, x.k + 3, k, nk, cg2, gm1h, kp);
      pin(kp);
    }
    cons_to_prim_fast(x.q, g, pn);
    axis_step<LIM>(st, pn, mr, kd, s - 1 >= 2 && s - 1 <= ni - 3, s >= 2 && s <= ni - 3, s >= 2 && s <= ni - 2,
                   s >= 2 && s <= ni - 1, cg2, gm1h, kp, out);
    if (s >= tl.p0 + 2 && own) {
#pragma unroll
      for (int v = 0; v < 5; ++v) at(b.fs + v * N, cell(s - 2)) = out[v];
    }
  }
}

// Both sweeps that march along i, one launch: neither needs the other, and
// waves of the one (loads, few chains) and of the other (FP64 chains) fill
// each other's waits on a SIMD.  Each wave its own tile of its sweep's table,
// no barrier; workgroups alternate between the sweeps in groups of eight (one
// to each XCD), so both spread over every XCD, each in its table's order.
template <int LIM>
__global__ void __launch_bounds__(SWEEP_NT) __attribute__((amdgpu_waves_per_eu(2)))
k_vjp_i(const BlockDesc* __restrict__ blocks, const SweepTile* __restrict__ sv, int nv,
        const SweepTile* __restrict__ sik, int nik, int stage, Gas gas, double dt) {
  __shared__ double rest[SW_N * SWEEP_NT];
  const int gv = (nv + 3) / 4, gik = (nik + 3) / 4, wg = (int)blockIdx.x, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int paired = 8 * ((gv < gik ? gv : gik) / 8);   // workgroups of each sweep that alternate
  const bool visc = wg < 2 * paired ? (wg >> 3) & 1 : wg - paired < gv;
  int idx;
  if (wg < 2 * paired) idx = (wg >> 4) * 8 + (wg & 7);
  else idx = visc ? wg - paired : wg - gv;
  if (visc) {
    const int t = xcd_remap(idx, gv) * 4 + w;
    if (t < nv) sweep_visc(blocks[sv[t].block], sv[t], stage, gas, dt);
  } else {
    const int t = xcd_remap(idx, gik) * 4 + w;
    if (t < nik) sweep_ik<LIM>(rest, blocks[sik[t].block], sik[t], stage, gas, dt);
  }
}

// The j axis, and what is left to do for a cell: lanes are 64 columns (i, k)
// from base on (k fastest), rows p0 .. p1-1.
template <int LIM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
k_vjp_j(const BlockDesc* __restrict__ blocks, const SweepTile* __restrict__ tiles, int ntiles, int stage, Gas gas,
        double dt) {
  const int w = xcd_remap(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w >= ntiles) return;
  const SweepTile tl = tiles[w];
  const BlockDesc& b = blocks[tl.block];
  const int lane = threadIdx.x & 63, nj = b.nj, nk = b.nk;
  const int64_t N = b.N;
  const unsigned njk = (unsigned)nj * (unsigned)nk, nik = (unsigned)b.ni * (unsigned)nk;
  const double *qs, *lin;
  double* lout;
  vjp_bufs(b, stage, qs, lin, lout);
  const double hcm = uniform(0.5 * stage_cmu(stage, dt * b.dt_scale));
  const double g = gas.gamma, cg2 = uniform(2.0 * g / (g - 1.0)), gm1h = uniform(0.5 * (g - 1.0));
  const unsigned cl = (unsigned)(tl.base + lane);
  const bool own = cl < nik;
  const unsigned cc = own ? cl : nik - 1u;
  const int i = (int)(cc / (unsigned)nk), k = (int)(cc % (unsigned)nk);
  const unsigned col = (unsigned)i * njk + (unsigned)k;
  auto cell = [&](int s) -> unsigned { return col + (unsigned)(s < 0 ? 0 : (s >= nj ? nj - 1 : s)) * (unsigned)nk; };

  __shared__ double rest[SW_N * SWEEP_NT];
  AxisSweep st;
  st.rest = rest + threadIdx.x;
  sweep_begin<LIM>(st, b, qs, lin, cell(tl.p0 - 3), cell(tl.p0 - 2), cell(tl.p0 - 1), 3, g, hcm);
  SweepLoads<3> x;
  for (int s = tl.p0 - 1; s <= tl.p1 + 1; ++s) {
    double pn[5], mr[5], kd[3], out[5], kp[5] = {0, 0, 0, 0, 0};
    sweep_load(x, b, qs, lin, cell(s), cell(s + 1), 3);
    const double r = hcm * rcp_hd(x.vol + 1e-300);
#pragma unroll
    for (int v = 0; v < 5; ++v) mr[v] = r * x.l[v];
#pragma unroll
    for (int m = 0; m < 3; ++m) kd[m] = x.k[m];
    cons_to_prim_fast(x.q, g, pn);
    axis_step<LIM>(st, pn, mr, kd, s - 1 >= 2 && s - 1 <= nj - 3, s >= 2 && s <= nj - 3, s >= 2 && s <= nj - 2,
                   s >= 2 && s <= nj - 1, cg2, gm1h, kp, out);
    if (s >= tl.p0 + 2 && own) {
      cell_vjp_finish(b, qs, lin, lout, s - 2, cell(s - 2), gas, stage, out);
    }
  }
}

// ---------------------------------------------------------------------------
// host launcher
// ---------------------------------------------------------------------------
void launch_stage_vjp(const BlockDesc* blocks, const SweepTile* sv, int nv, const SweepTile* sik, int nik,
                      const SweepTile* sj, int nsj, int stage, const Gas& gas, double dt, int lim, hipStream_t st) {
  const unsigned wi = (unsigned)((nv + 3) / 4 + (nik + 3) / 4), wj = (unsigned)((nsj + 3) / 4);
  if (lim == LIM_VANLEER) {
    k_vjp_i<LIM_VANLEER><<<wi, SWEEP_NT, 0, st>>>(blocks, sv, nv, sik, nik, stage, gas, dt);
    k_vjp_j<LIM_VANLEER><<<wj, SWEEP_NT, 0, st>>>(blocks, sj, nsj, stage, gas, dt);
  } else {
    k_vjp_i<LIM_MINMOD><<<wi, SWEEP_NT, 0, st>>>(blocks, sv, nv, sik, nik, stage, gas, dt);
    k_vjp_j<LIM_MINMOD><<<wj, SWEEP_NT, 0, st>>>(blocks, sj, nsj, stage, gas, dt);
  }
}

}  // namespace famrdp

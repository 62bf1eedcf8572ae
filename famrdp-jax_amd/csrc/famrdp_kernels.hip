// FP64 kernels of famrdp_jax's RHS + TVD-RK3 path for gfx950.
//
// Kernel families:
//   * unit kernels behind the reference's pointwise API (eos, MUSCL-2, Roe);
//   * the direct stage pair (viscous flux tensor, then inviscid + viscous
//     divergence + RK3 combination), one thread per padded cell, in a
//     per-block form and a batched form driven by a tile table;
//   * halo gather/scatter (pre-exchange semantics) and ghost-cell BC faces;
//   * grid metrics and the CFL / positivity reduction.
#include "famrdp_kernels.h"
#include "famrdp_ghost.h"
#include "famrdp_tiles.h"

namespace famrdp {

// ---------------------------------------------------------------------------
// Unit kernels
// ---------------------------------------------------------------------------

__global__ void k_cons_to_prim(const double* __restrict__ q, double* __restrict__ pv, int64_t n, double g) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  double a[5], b[5];
  for (int v = 0; v < 5; ++v) a[v] = q[v * n + t];
  cons_to_prim(a, g, b);
  for (int v = 0; v < 5; ++v) pv[v * n + t] = b[v];
}

__global__ void k_prim_to_cons(const double* __restrict__ pv, double* __restrict__ q, int64_t n, double g) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  double a[5], b[5];
  for (int v = 0; v < 5; ++v) a[v] = pv[v * n + t];
  prim_to_cons(a, g, b);
  for (int v = 0; v < 5; ++v) q[v * n + t] = b[v];
}

__global__ void k_sutherland(const double* __restrict__ T, double* __restrict__ mu, int64_t n, double mu0,
                             double T0, double Ts) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) mu[t] = sutherland(T[t], mu0, T0, Ts);
}

__global__ void k_speed_of_sound(const double* __restrict__ rho, const double* __restrict__ p,
                                 double* __restrict__ c, int64_t n, double g) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) c[t] = sqrt(g * p[t] / rho[t]);
}

__global__ void k_limiter(const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ out,
                          int64_t n, int lim) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) out[t] = limit(lim, a[t], b[t]);
}

// pv (nvar, n0, n1, n2); faces along `axis` (1..3) -> (nvar, ..., n_axis-3, ...)
__global__ void k_muscl2(const double* __restrict__ pv, double* __restrict__ pL, double* __restrict__ pR,
                         int nvar, int n0, int n1, int n2, int axis, int lim) {
  const int f0 = axis == 1 ? n0 - 3 : n0, f1 = axis == 2 ? n1 - 3 : n1, f2 = axis == 3 ? n2 - 3 : n2;
  const int64_t nf = (int64_t)f0 * f1 * f2;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nf) return;
  const int a2 = (int)(t % f2), a1 = (int)((t / f2) % f1), a0 = (int)(t / ((int64_t)f2 * f1));
  const int64_t s0 = (int64_t)n1 * n2, s1 = n2;
  const int64_t stride = axis == 1 ? s0 : (axis == 2 ? s1 : 1);
  // face f along the axis sits between cells f+1 and f+2: base cell index = f
  const int64_t base = (int64_t)a0 * s0 + (int64_t)a1 * s1 + a2;
  const int64_t N = (int64_t)n0 * n1 * n2;
  for (int v = 0; v < nvar; ++v) {
    const double* p = pv + v * N + base;
    const double pmm = p[0], pc = p[stride], pp1 = p[2 * stride], pp2 = p[3 * stride];
    const double sL = limit(lim, pc - pmm, pp1 - pc);
    const double sR = limit(lim, pp1 - pc, pp2 - pp1);
    pL[v * nf + t] = pc + 0.5 * sL;
    pR[v * nf + t] = pp1 - 0.5 * sR;
  }
}

__global__ void k_roe_flux(const double* __restrict__ UL, const double* __restrict__ UR,
                           const double* __restrict__ nx, double* __restrict__ F, int64_t n, double g,
                           double eps_entropy) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  double a[5], b[5], nn[3], f[5];
  for (int v = 0; v < 5; ++v) { a[v] = UL[v * n + t]; b[v] = UR[v * n + t]; }
  for (int v = 0; v < 3; ++v) nn[v] = nx[v * n + t];
  roe_flux(a, b, nn, g, eps_entropy, f);
  for (int v = 0; v < 5; ++v) F[v * n + t] = f[v];
}

// ---------------------------------------------------------------------------
// Direct stage: per-cell device functions
// ---------------------------------------------------------------------------

// Viscous flux tensor G at cell c (rhs/viscous.py:30-108, roll wrap).
__device__ __forceinline__ void cell_viscous_flux(const double* __restrict__ q, const double* __restrict__ kxyz,
                                                  double* __restrict__ G, int ni, int nj, int nk, int64_t N,
                                                  int64_t c, const Gas& gas) {
  const int k = (int)(c % nk), j = (int)((c / nk) % nj), i = (int)(c / ((int64_t)nk * nj));
  const int64_t sj = nk, si = (int64_t)nj * nk;
  const int64_t cm[3] = {c + (wrap_m(i, ni) - i) * si, c + (wrap_m(j, nj) - j) * sj, c + (wrap_m(k, nk) - k)};
  const int64_t cp[3] = {c + (wrap_p(i, ni) - i) * si, c + (wrap_p(j, nj) - j) * sj, c + (wrap_p(k, nk) - k)};
  double pv[5];
  load_prim(q, N, c, gas.gamma, pv);
  const double T = temperature(pv, gas.R);
  double d[3][4];
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    double pp[5], pm[5];
    load_prim(q, N, cp[l], gas.gamma, pp);
    load_prim(q, N, cm[l], gas.gamma, pm);
    d[l][0] = 0.5 * (pp[1] - pm[1]);
    d[l][1] = 0.5 * (pp[2] - pm[2]);
    d[l][2] = 0.5 * (pp[3] - pm[3]);
    d[l][3] = 0.5 * (temperature(pp, gas.R) - temperature(pm, gas.R));
  }
  double kk[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) kk[m] = kxyz[m * N + c];
  double g9[9];
  viscous_flux(pv, T, d, kk, gas, g9);
#pragma unroll
  for (int m = 0; m < 9; ++m) G[m * N + c] = g9[m];
}

// Inviscid RHS at cell c (rhs/invscd.py:53-131): axis contributions added in
// axis order, only where 2 <= c_d <= n_d - 3.
__device__ __forceinline__ void cell_invscd(const double* __restrict__ q, const double* __restrict__ kxyz,
                                            const double* __restrict__ vol, int ni, int nj, int nk, int64_t N,
                                            int64_t c, double g, int lim, double inv[5]) {
  const int k = (int)(c % nk), j = (int)((c / nk) % nj), i = (int)(c / ((int64_t)nk * nj));
  const int idx[3] = {i, j, k};
  const int n[3] = {ni, nj, nk};
  const int64_t st[3] = {(int64_t)nj * nk, nk, 1};
#pragma unroll
  for (int v = 0; v < 5; ++v) inv[v] = 0.0;
  const double rvol = vol[c] + 1e-300;
  for (int d = 0; d < 3; ++d) {
    if (idx[d] < 2 || idx[d] > n[d] - 3) continue;
    double pv[5][5];
#pragma unroll
    for (int s = 0; s < 5; ++s) load_prim(q, N, c + (s - 2) * st[d], g, pv[s]);
    double kd[3][3];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int m = 0; m < 3; ++m) kd[s][m] = kxyz[(d * 3 + m) * N + c + (s - 1) * st[d]];
    double Fm[5], Fp[5];
    face_flux(pv[0], pv[1], pv[2], pv[3], kd[0], kd[1], g, lim, Fm);   // face c-1/2
    face_flux(pv[1], pv[2], pv[3], pv[4], kd[1], kd[2], g, lim, Fp);   // face c+1/2
#pragma unroll
    for (int v = 0; v < 5; ++v) inv[v] = inv[v] + (-(Fp[v] - Fm[v]) / rvol);
  }
}

// Viscous divergence at cell c from G (rhs/viscous.py:86-108): for each row,
// sum over j of sum_l kxyz[l, j] * 0.5 (G_j(+e_l) - G_j(-e_l)).
__device__ __forceinline__ void cell_viscous_div(const double* __restrict__ G, const double* __restrict__ kxyz,
                                                 int ni, int nj, int nk, int64_t N, int64_t c, double vis[4]) {
  const int k = (int)(c % nk), j = (int)((c / nk) % nj), i = (int)(c / ((int64_t)nk * nj));
  const int64_t sj = nk, si = (int64_t)nj * nk;
  const int64_t cm[3] = {c + (wrap_m(i, ni) - i) * si, c + (wrap_m(j, nj) - j) * sj, c + (wrap_m(k, nk) - k)};
  const int64_t cp[3] = {c + (wrap_p(i, ni) - i) * si, c + (wrap_p(j, nj) - j) * sj, c + (wrap_p(k, nk) - k)};
  double kk[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) kk[m] = kxyz[m * N + c];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    double res = 0.0;
#pragma unroll
    for (int jj = 0; jj < 3; ++jj) {
      const double* Gc = G + gidx(r, jj) * N;
      const double d0 = 0.5 * (Gc[cp[0]] - Gc[cm[0]]);
      const double d1 = 0.5 * (Gc[cp[1]] - Gc[cm[1]]);
      const double d2 = 0.5 * (Gc[cp[2]] - Gc[cm[2]]);
      res = res + (d0 * kk[0 * 3 + jj] + d1 * kk[1 * 3 + jj] + d2 * kk[2 * 3 + jj]);
    }
    vis[r] = res;
  }
}

// Shu-Osher combination (solver/step.py:45-53).
__device__ __forceinline__ double rk_combine(int stage, double q0, double qs, double dt, double r) {
  if (stage == 1) return qs + dt * r;
  if (stage == 2) return 0.75 * q0 + 0.25 * (qs + dt * r);
  return (1.0 / 3.0) * q0 + (2.0 / 3.0) * (qs + dt * r);
}

// q0 may alias qout (stage 3 writes the state in place): both are read for
// cell c only, and every read happens before the first write.
__device__ __forceinline__ void cell_stage(const double* __restrict__ qin, const double* q0, double* qout,
                                           const double* __restrict__ kxyz, const double* __restrict__ vol,
                                           const double* __restrict__ G, int ni, int nj, int nk, int64_t N, int64_t c,
                                           double g, int lim, double dt, int stage) {
  double inv[5], vis[4];
  cell_invscd(qin, kxyz, vol, ni, nj, nk, N, c, g, lim, inv);
  cell_viscous_div(G, kxyz, ni, nj, nk, N, c, vis);
  double rhs[5];
  rhs[0] = inv[0] + 0.0;
  rhs[1] = inv[1] + vis[0];
  rhs[2] = inv[2] + vis[1];
  rhs[3] = inv[3] + vis[2];
  rhs[4] = inv[4] + vis[3];
  double qs[5], qq0[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    qs[v] = qin[v * N + c];
    qq0[v] = stage == 1 ? 0.0 : q0[v * N + c];
  }
#pragma unroll
  for (int v = 0; v < 5; ++v) qout[v * N + c] = rk_combine(stage, qq0[v], qs[v], dt, rhs[v]);
}

// ---------------------------------------------------------------------------
// Direct stage kernels: per-block launches
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_viscous_flux(const double* __restrict__ q, const double* __restrict__ kxyz,
                                                      double* __restrict__ G, int ni, int nj, int nk, Gas gas) {
  const int64_t N = (int64_t)ni * nj * nk;
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c < N) cell_viscous_flux(q, kxyz, G, ni, nj, nk, N, c, gas);
}

__global__ void k_fastmath_probe(const double* __restrict__ x, double* __restrict__ r, double* __restrict__ s,
                                 double* __restrict__ q, int64_t n) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) {
    r[t] = rcp(x[t]);
    s[t] = fsqrt(x[t]);
    if (q) q[t] = rsq_acc(x[t]);
  }
}

__global__ void k_fastmath_probe1(const double* __restrict__ x, double* __restrict__ r, double* __restrict__ q,
                                  int64_t n) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t < n) {
    r[t] = rcp1(x[t]);
    q[t] = rsq1(x[t]);
  }
}

__global__ void __launch_bounds__(256) k_stage(const double* __restrict__ qin, const double* q0,
                                               double* qout, const double* __restrict__ kxyz,
                                               const double* __restrict__ vol, const double* __restrict__ G, int ni,
                                               int nj, int nk, double g, int lim, double dt, int stage) {
  const int64_t N = (int64_t)ni * nj * nk;
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c < N) cell_stage(qin, q0, qout, kxyz, vol, G, ni, nj, nk, N, c, g, lim, dt, stage);
}

__global__ void k_axpby(double* __restrict__ out, double a, const double* __restrict__ x, double b,
                        const double* __restrict__ y, double c, const double* __restrict__ z, int64_t n, int mode) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= n) return;
  out[t] = mode == 1 ? y[t] + c * z[t] : a * x[t] + b * (y[t] + c * z[t]);
}

// ---------------------------------------------------------------------------
// Batched direct stage kernels: persistent grid over a tile table that spans
// every block of the plan (the block-offset table is `blocks`).
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_viscous_flux_batched(const BlockDesc* __restrict__ blocks,
                                                              const Tile* __restrict__ tiles, int ntiles, int stage,
                                                              Gas gas) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const BlockDesc& b = blocks[tl.block];
    const int64_t c = (int64_t)tl.start + threadIdx.x;
    if (c < b.N) {
      const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
      Gas gb = gas;
      gb.mu0 = b.mu0;
      cell_viscous_flux(qin, b.kxyz, b.G, b.ni, b.nj, b.nk, b.N, c, gb);
    }
  }
}

__global__ void __launch_bounds__(256) k_stage_batched(const BlockDesc* __restrict__ blocks,
                                                       const Tile* __restrict__ tiles, int ntiles, double g, int lim,
                                                       double dt, int stage) {
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const BlockDesc& b = blocks[tl.block];
    const int64_t c = (int64_t)tl.start + threadIdx.x;
    if (c < b.N) {
      const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
      double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
      cell_stage(qin, b.q, qout, b.kxyz, b.vol, b.G, b.ni, b.nj, b.nk, b.N, c, g, lim, dt * b.dt_scale, stage);
    }
  }
}

// ---------------------------------------------------------------------------
// Halo exchange (mesh/halo.py:56-92): gather every final ghost value from the
// pre-exchange state into `stage`, then scatter; two launches give the
// reference's "all copies read the original arrays" semantics.
// ---------------------------------------------------------------------------

__global__ void k_halo_gather(const BlockDesc* __restrict__ blocks, const HaloEntry* __restrict__ e, int n,
                              double* __restrict__ stage) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const HaloEntry h = e[t];
  const BlockDesc s = blocks[h.sb];
#pragma unroll
  for (int v = 0; v < 5; ++v) stage[(int64_t)v * n + t] = s.q[v * s.N + h.sc];
}

__global__ void k_halo_scatter(const BlockDesc* __restrict__ blocks, const HaloEntry* __restrict__ e, int n,
                               const double* __restrict__ stage) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const HaloEntry h = e[t];
  const BlockDesc b = blocks[h.tb];
#pragma unroll
  for (int v = 0; v < 5; ++v) b.q[v * b.N + h.tc] = stage[(int64_t)v * n + t];
}

// ---------------------------------------------------------------------------
// Ghost-cell BCs on their own (physics/bc/*.py).  One launch per face index
// (Face order), covering that face of every block that has a BC there;
// blockIdx.y = entry.
// ---------------------------------------------------------------------------

__global__ void k_bc_face(const BlockDesc* __restrict__ blocks, const BcEntry* __restrict__ entries, int ghost,
                          double gamma, double R) {
  const BcEntry e = entries[blockIdx.y];
  const BlockDesc b = blocks[e.block];
  const int ax = e.face / 2;            // 0: i, 1: j, 2: k
  const int na = ax == 0 ? b.ni : (ax == 1 ? b.nj : b.nk);
  const int64_t sj = b.nk, si = (int64_t)b.nj * b.nk;
  const int64_t sa = ax == 0 ? si : (ax == 1 ? sj : (int64_t)1);
  const int n1 = ax == 0 ? b.nj : b.ni, n2 = ax == 2 ? b.nj : b.nk;
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= (int64_t)n1 * n2) return;
  const int64_t base = (t / n2) * (ax == 0 ? sj : si) + (t % n2) * (ax == 2 ? sj : (int64_t)1);
  for (int gl = 0; gl < ghost; ++gl) {
    int outer, inner;
    bc_pair(e, ghost, na, gl, outer, inner);
    const int64_t co = base + outer * sa, ci = base + inner * sa;
    double q[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = b.q[v * b.N + ci];
    bc_apply(e, gamma, R, q);
#pragma unroll
    for (int v = 0; v < 5; ++v) b.q[v * b.N + co] = q[v];
  }
}

// ---------------------------------------------------------------------------
// Ghost cells of a step (famrdp_ghost.h): 20 bytes of table and 80 of state an
// entry, in one launch or two, where the exchange and the faces one after the
// other were up to eight (55 x 55 x 15 free stream all around: 36 us, now 4).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void ghost_chain(const GhostChain* __restrict__ chains, const BcEntry* __restrict__ ops,
                                            int chain, double gamma, double R, double q[5]) {
  if (chain > 0) {
    const GhostChain& c = chains[chain];
    for (int i = 0; i < c.n; ++i) bc_apply(ops[c.op[i]], gamma, R, q);
  }
}

__device__ __forceinline__ void ghost_value(const BlockDesc* __restrict__ blocks, const GhostChain* __restrict__ chains,
                                            const BcEntry* __restrict__ ops, int sb, int sc, int chain, double gamma,
                                            double R, double q[5]) {
  if (sb >= 0) {
    const BlockDesc& s = blocks[sb];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = s.q[v * s.N + sc];
  } else {
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = 0.0;   // replaced by the chain's free stream
  }
  ghost_chain(chains, ops, chain, gamma, R, q);
}

// Direct entries, then the staged ones into the staging buffer, then the
// recorded values.
__global__ void __launch_bounds__(256) k_ghost_first(const BlockDesc* __restrict__ blocks,
                                                     const GhostEntry* __restrict__ e, int ndirect, int nstaged,
                                                     const GhostChain* __restrict__ chains,
                                                     const BcEntry* __restrict__ ops, double gamma, double R,
                                                     double* __restrict__ stage, const GhostSnap* __restrict__ snaps,
                                                     int nsnap, SnapPtrs snap) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  double q[5];
  if (t < ndirect + nstaged) {
    const GhostEntry h = e[t];
    ghost_value(blocks, chains, ops, h.sb, h.sc, h.chain, gamma, R, q);
    if (t < ndirect) {
      const BlockDesc& b = blocks[h.tb];
#pragma unroll
      for (int v = 0; v < 5; ++v) b.q[v * b.N + h.tc] = q[v];
    } else {
#pragma unroll
      for (int v = 0; v < 5; ++v) stage[(int64_t)v * nstaged + (t - ndirect)] = q[v];
    }
  } else if (t < ndirect + nstaged + nsnap) {
    const GhostSnap h = snaps[t - ndirect - nstaged];
    ghost_value(blocks, chains, ops, h.sb, h.sc, h.chain, gamma, R, q);
    double* dst = snap.face[h.face] + h.off;
#pragma unroll
    for (int v = 0; v < 5; ++v) dst[v * h.stride] = q[v];
  }
}

// The staged entries from the staging buffer, and the direct ones whose target
// a staged entry or a record had to read first.
__global__ void __launch_bounds__(256) k_ghost_second(const BlockDesc* __restrict__ blocks,
                                                      const GhostEntry* __restrict__ e, int nstaged, int nlate,
                                                      const GhostChain* __restrict__ chains,
                                                      const BcEntry* __restrict__ ops, double gamma, double R,
                                                      const double* __restrict__ stage) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nstaged + nlate) return;
  const GhostEntry h = e[t];
  double q[5];
  if (t < nstaged) {
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = stage[(int64_t)v * nstaged + t];
  } else {
    ghost_value(blocks, chains, ops, h.sb, h.sc, h.chain, gamma, R, q);
  }
  const BlockDesc& b = blocks[h.tb];
#pragma unroll
  for (int v = 0; v < 5; ++v) b.q[v * b.N + h.tc] = q[v];
}

// ---------------------------------------------------------------------------
// Grid metrics (mesh/metric.py:18-70): 4th-order central differences with
// roll wrap, J[m][l] = dx_m/dxi_l, jac = det J, kxyz = inv(J) as [l][m].
// The floor is HBM (112 bytes a cell); what held it up were the 36 loads a
// cell, every wave's at 16 cycles of a CU's address unit.  So a workgroup
// holds TJ x TK columns (a thread each) and walks planes along i: the five
// planes of the i difference stay in registers, a plane with two cells around
// it lies in LDS for the other two, and a cell takes three loads and its share
// of the halo's (small and thin grids are left to a thread per cell:
// metrics_marched).  The next plane's loads are issued before a plane is worked
// on; two LDS planes in turn leave one barrier a plane.  164 x 132 x 148 cells
// 100 us (127 with a thread per cell), 204^3 318 (363), 264^3 613 (755): what
// is left are the eleven streams it writes.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int roll(int i, int n) {
  const int r = i % n;
  return r < 0 ? r + n : r;
}

constexpr int METRIC_TJ = 8, METRIC_TK = 32;

// jac, vol and kxyz of cell c from its Jacobian
__device__ __forceinline__ void metrics_of(const double J[3][3], int64_t c, int64_t N, double* __restrict__ jac,
                                           double* __restrict__ kxyz, double* __restrict__ vol) {
  const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
  const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
  const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
  const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
  const double inv[3][3] = {
      {c00 / det, (J[0][2] * J[2][1] - J[0][1] * J[2][2]) / det, (J[0][1] * J[1][2] - J[0][2] * J[1][1]) / det},
      {c01 / det, (J[0][0] * J[2][2] - J[0][2] * J[2][0]) / det, (J[0][2] * J[1][0] - J[0][0] * J[1][2]) / det},
      {c02 / det, (J[0][1] * J[2][0] - J[0][0] * J[2][1]) / det, (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / det}};
  jac[c] = det;
  vol[c] = fabs(det);
  for (int l = 0; l < 3; ++l)
    for (int m = 0; m < 3; ++m) kxyz[(l * 3 + m) * N + c] = inv[l][m];
}

// Whether a grid is marched in tiles: where there are cells enough (below, the
// segments' first planes cost more than the loads they save: 36^3 cells 6.2 us
// marched, 5.0 a thread per cell; 60^3 9.8 and 11.0; 120,000 of 33 along k 9.3
// and 7.1, 400,000 of 24 13.7 and 16) and the tiles' columns are not too many for
// the block's (columns past it take their share of the time: at 10^6 cells of 18
// along k, 1.8 times the columns, 30 us both; of 16, twice, 33 and 28.5; of 9,
// 3.6 times, 49 and 31; of 1, 32 times, 359 and 29).  Large grids, bound by
// memory, bear more: 8 * 10^6 cells of 16 262 and 306, of 14, 2.3 times, 309 both.
inline bool metrics_marched(int ni, int nj, int nk) {
  const int64_t N = (int64_t)ni * nj * nk;
  const double columns = (double)((nj + METRIC_TJ - 1) / METRIC_TJ * METRIC_TJ) *
                         (double)((nk + METRIC_TK - 1) / METRIC_TK * METRIC_TK) / ((double)nj * nk);
  return N >= (1 << 17) && columns <= (N < (1 << 18) ? 1.2 : (N < (1 << 22) ? 1.9 : 2.3));
}

// The others: a thread per cell.
__global__ void __launch_bounds__(256) k_metrics_cell(const double* __restrict__ xyz, double* __restrict__ jac,
                                                      double* __restrict__ kxyz, double* __restrict__ vol, int ni, int nj,
                                                      int nk) {
  const int64_t N = (int64_t)ni * nj * nk;
  const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (c >= N) return;
  const int k = (int)(c % nk), j = (int)((c / nk) % nj), i = (int)(c / ((int64_t)nk * nj));
  const int idx[3] = {i, j, k}, n[3] = {ni, nj, nk};
  const int64_t st[3] = {(int64_t)nj * nk, nk, 1};
  double J[3][3];
  for (int l = 0; l < 3; ++l) {
    int64_t o[5];
    for (int s = -2; s <= 2; ++s) o[s + 2] = c + (int64_t)(roll(idx[l] + s, n[l]) - idx[l]) * st[l];
    for (int m = 0; m < 3; ++m) {
      const double* f = xyz + m * N;
      J[m][l] = (-f[o[4]] + 8.0 * f[o[3]] - 8.0 * f[o[1]] + f[o[0]]) / 12.0;
    }
  }
  metrics_of(J, c, N, jac, kxyz, vol);
}

// Workgroups: (segment of len planes, tile), the tile index fastest.
__global__ void __launch_bounds__(METRIC_TJ * METRIC_TK) __attribute__((amdgpu_waves_per_eu(4))) k_metrics(const double* __restrict__ xyz,
                                                                   double* __restrict__ jac, double* __restrict__ kxyz,
                                                                   double* __restrict__ vol, int ni, int nj, int nk,
                                                                   int len) {
  constexpr int TJ = METRIC_TJ, TK = METRIC_TK, W = TK + 4, P = (TJ + 4) * W, HJ = 4 * TK, H = HJ + 4 * TJ;
  static_assert(H <= TJ * TK, "a thread per halo cell");
  __shared__ double lds[2][3][P];
  const int t = threadIdx.x, tj = t / TK, tk = t % TK;
  const int ntk = (nk + TK - 1) / TK, ntj = (nj + TJ - 1) / TJ;
  const int wg = xcd_remap(blockIdx.x, gridDim.x), tile = wg % (ntj * ntk), seg = wg / (ntj * ntk);
  const int j0 = tile / ntk * TJ, k0 = tile % ntk * TK;
  const int iA = seg * len, iB = min(iA + len, ni);
  const int64_t N = (int64_t)ni * nj * nk, si = (int64_t)nj * nk;
  const bool own = j0 + tj < nj && k0 + tk < nk;
  const int64_t col = (int64_t)roll(j0 + tj, nj) * nk + roll(k0 + tk, nk);
  const int slot = (tj + 2) * W + tk + 2;
  // the thread's halo cell: rows -2, -1, TJ, TJ + 1, then columns likewise
  int hj = 0, hk = 0;
  if (t < HJ) {
    const int e = t / TK;
    hj = e < 2 ? e - 2 : TJ + e - 2;
    hk = t % TK;
  } else if (t < H) {
    const int e = (t - HJ) / TJ;
    hj = (t - HJ) % TJ;
    hk = e < 2 ? e - 2 : TK + e - 2;
  }
  const int64_t hcol = (int64_t)roll(j0 + hj, nj) * nk + roll(k0 + hk, nk);
  const int hslot = (hj + 2) * W + hk + 2;
  double f[3][5], h[3];                  // planes i-2 .. i+2 of the column; the halo cell on plane i
#pragma unroll
  for (int m = 0; m < 3; ++m) {
#pragma unroll
    for (int p = 0; p < 4; ++p) f[m][p + 1] = xyz[m * N + roll(iA + p - 2, ni) * si + col];
    h[m] = xyz[m * N + iA * si + hcol];
  }
  double nf[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) nf[m] = xyz[m * N + roll(iA + 2, ni) * si + col];
  for (int i = iA; i < iB; ++i) {
    double (*s)[P] = lds[(i - iA) & 1];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
#pragma unroll
      for (int p = 0; p < 4; ++p) f[m][p] = f[m][p + 1];
      f[m][4] = nf[m];
      s[m][slot] = f[m][2];
      if (t < H) s[m][hslot] = h[m];
    }
    __syncthreads();
    const int64_t pn = roll(i + 3, ni) * si, ph = roll(i + 1, ni) * si;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      nf[m] = xyz[m * N + pn + col];
      h[m] = xyz[m * N + ph + hcol];
    }
    double J[3][3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double* c = s[m] + slot;
      J[m][0] = (-f[m][4] + 8.0 * f[m][3] - 8.0 * f[m][1] + f[m][0]) / 12.0;
      J[m][1] = (-c[2 * W] + 8.0 * c[W] - 8.0 * c[-W] + c[-2 * W]) / 12.0;
      J[m][2] = (-c[2] + 8.0 * c[1] - 8.0 * c[-1] + c[-2]) / 12.0;
    }
    if (own) metrics_of(J, i * si + col, N, jac, kxyz, vol);
  }
}

// ---------------------------------------------------------------------------
// CFL time step and positivity monitor over interior cells (two passes, no
// atomics): per-workgroup max spectral radius and bad-cell count, then one
// workgroup reduces them.
// ---------------------------------------------------------------------------

// coordinates of cell c of an (., nj, nk) block; 32-bit divisions where c has
// no more (the same for a whole launch: N decides).  k_cfl_partial reads 120
// bytes a cell; on 164 x 132 x 148 cells 64-bit divisions held it at 90 us, 79
// without.
__device__ __forceinline__ void cell_coords(int64_t c, int64_t N, int nj, int nk, int& i, int& j, int& k) {
  if (N <= INT32_MAX) {
    const unsigned u = (unsigned)c, r = u / (unsigned)nk, p = r / (unsigned)nj;
    k = (int)(u - r * (unsigned)nk);
    j = (int)(r - p * (unsigned)nj);
    i = (int)p;
  } else {
    k = (int)(c % nk);
    j = (int)((c / nk) % nj);
    i = (int)(c / ((int64_t)nk * nj));
  }
}

__global__ void __launch_bounds__(256) k_cfl_partial(const double* __restrict__ q, const double* __restrict__ kxyz,
                                                     const double* __restrict__ vol, int ni, int nj, int nk, int ghost,
                                                     Gas gas, double* __restrict__ part_lam,
                                                     double* __restrict__ part_bad) {
  __shared__ double slam[256];
  __shared__ double sbad[256];
  const int64_t N = (int64_t)ni * nj * nk;
  const int ii = ni - 2 * ghost, jj = nj - 2 * ghost, kk = nk - 2 * ghost;
  const int64_t nint = (int64_t)ii * jj * kk;
  double lam = 0.0, bad = 0.0;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < nint; t += (int64_t)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_coords(t, nint, jj, kk, i, j, k);
    i += ghost; j += ghost; k += ghost;
    const int64_t c = ((int64_t)i * nj + j) * nk + k;
    double pv[5];
    load_prim(q, N, c, gas.gamma, pv);
    const bool ok = isfinite(pv[0]) && isfinite(pv[1]) && isfinite(pv[2]) && isfinite(pv[3]) && isfinite(pv[4]) &&
                    pv[0] > 0.0 && pv[4] > 0.0;
    if (!ok) { bad += 1.0; continue; }
    const double cs = sqrt(gas.gamma * pv[4] / pv[0]);
    const double T = pv[4] / (pv[0] * gas.R);
    const double mu = sutherland(T, gas.mu0, gas.T0, gas.Ts);
    double inv = 0.0, ksq = 0.0;
    for (int d = 0; d < 3; ++d) {
      const double k0 = kxyz[(d * 3 + 0) * N + c], k1 = kxyz[(d * 3 + 1) * N + c], k2 = kxyz[(d * 3 + 2) * N + c];
      const double kn2 = k0 * k0 + k1 * k1 + k2 * k2;
      inv = inv + (fabs(pv[1] * k0 + pv[2] * k1 + pv[3] * k2) + cs * sqrt(kn2));
      ksq = ksq + kn2;
    }
    const double l = inv / vol[c] + fmax(4.0 / 3.0, gas.gamma / gas.Pr_lam) * mu / pv[0] * ksq;
    lam = fmax(lam, l);
  }
  slam[threadIdx.x] = lam;
  sbad[threadIdx.x] = bad;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      slam[threadIdx.x] = fmax(slam[threadIdx.x], slam[threadIdx.x + s]);
      sbad[threadIdx.x] += sbad[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part_lam[blockIdx.x] = slam[0];
    part_bad[blockIdx.x] = sbad[0];
  }
}

__global__ void __launch_bounds__(256) k_cfl_final(const double* __restrict__ part_lam,
                                                   const double* __restrict__ part_bad, int n, double cfl,
                                                   double* __restrict__ out) {
  __shared__ double slam[256];
  __shared__ double sbad[256];
  double lam = 0.0, bad = 0.0;
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    lam = fmax(lam, part_lam[t]);
    bad += part_bad[t];
  }
  slam[threadIdx.x] = lam;
  sbad[threadIdx.x] = bad;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      slam[threadIdx.x] = fmax(slam[threadIdx.x], slam[threadIdx.x + s]);
      sbad[threadIdx.x] += sbad[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = cfl / slam[0];
    out[1] = slam[0];
    out[2] = sbad[0];
  }
}

// ---------------------------------------------------------------------------
// Start of a step that leaves its input alone: the states of up to
// STEP_START_BLOCKS blocks go into the arrays the step works in, and their
// descriptors into the plan's block table, both from the launch's arguments.
// Bound by HBM (80 bytes per cell); on a small block by the launch.
// ---------------------------------------------------------------------------
constexpr int STEP_START_BLOCKS = 16;
struct StepStart {
  BlockDesc block[STEP_START_BLOCKS];      // 16 of 136 bytes: within the 4 KB of a launch's arguments
  const double* src[STEP_START_BLOCKS];
};
static_assert(sizeof(StepStart) <= 3072, "launch arguments");

// A plan of no more blocks: the interior by the plan's tiles of 256 cells, a
// cell per thread, then the ghost cells by the ghost table's entries.  The
// entries' sources are values of before the exchange, which the input arrays
// keep, so what takes two launches in place (k_ghost_first, k_ghost_second)
// is part of this one: 20^3 cells 4.0 us, with the copy apart 9.6 in three.
__global__ void __launch_bounds__(256) k_step_start(const StepStart s, BlockDesc* __restrict__ blocks, int nblocks,
                                                    const Tile* __restrict__ tiles, int ntiles, int ghost,
                                                    const GhostEntry* __restrict__ e, int nentries,
                                                    const GhostChain* __restrict__ chains,
                                                    const BcEntry* __restrict__ ops, double gamma, double R) {
  if (blockIdx.x == 0 && (int)threadIdx.x < nblocks) blocks[threadIdx.x] = s.block[threadIdx.x];
  double q[5];
  if ((int)blockIdx.x < ntiles) {
    const Tile tl = tiles[blockIdx.x];
    const BlockDesc& d = s.block[tl.block];
    const int64_t c = (int64_t)tl.start + threadIdx.x;
    if (c >= d.N) return;
    const int r = (int)c / d.nk, k = (int)c - r * d.nk, i = r / d.nj, j = r - i * d.nj;   // (c < 2^31 in a plan)
    if (i < ghost || j < ghost || k < ghost || i >= d.ni - ghost || j >= d.nj - ghost || k >= d.nk - ghost) return;
    const double* src = s.src[tl.block];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = src[v * d.N + c];
#pragma unroll
    for (int v = 0; v < 5; ++v) d.q[v * d.N + c] = q[v];
    return;
  }
  const int t = ((int)blockIdx.x - ntiles) * 256 + (int)threadIdx.x;
  if (t >= nentries) return;
  const GhostEntry h = e[t];
#pragma unroll
  for (int v = 0; v < 5; ++v) q[v] = 0.0;   // a chain without a source starts with a free stream
  if (h.sb >= 0) {
    const int64_t N = s.block[h.sb].N;
    const double* src = s.src[h.sb];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = src[v * N + h.sc];
  }
  ghost_chain(chains, ops, h.chain, gamma, R, q);
  const BlockDesc& d = s.block[h.tb];
#pragma unroll
  for (int v = 0; v < 5; ++v) d.q[v * d.N + h.tc] = q[v];
}

// A share of the blocks of a larger plan, whole arrays (16-byte accesses where
// both allow); the exchange follows in place.  Grid: (chunks, blocks).
__global__ void __launch_bounds__(256) k_step_copy(const StepStart s, BlockDesc* __restrict__ blocks) {
  const BlockDesc& d = s.block[blockIdx.y];
  const double* __restrict__ src = s.src[blockIdx.y];
  double* __restrict__ dst = d.q;
  const int64_t n = 5 * d.N, step = (int64_t)gridDim.x * blockDim.x;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if ((((uintptr_t)src | (uintptr_t)dst) & 15) == 0) {
    const double2* __restrict__ s2 = (const double2*)src;
    double2* __restrict__ d2 = (double2*)dst;
    for (int64_t i = t; i < n / 2; i += step) d2[i] = s2[i];
    if ((n & 1) && t == 0) dst[n - 1] = src[n - 1];
  } else {
    for (int64_t i = t; i < n; i += step) dst[i] = src[i];
  }
  if (t == 0) blocks[blockIdx.y] = d;
}

// ---------------------------------------------------------------------------
// State monitor (Config.nan_check): interior cells of every block of a plan
// with a non-finite conservative value, rho <= 0 or p <= 0, counted per
// workgroup over the plan's tile table (no atomics), then summed.
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_monitor_partial(const BlockDesc* __restrict__ blocks,
                                                         const Tile* __restrict__ tiles, int ntiles, int ghost,
                                                         double gamma, double* __restrict__ part) {
  __shared__ double sbad[256];
  double bad = 0.0;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const Tile tl = tiles[t];
    const BlockDesc& b = blocks[tl.block];
    const int64_t c = (int64_t)tl.start + threadIdx.x;
    if (c >= b.N) continue;
    const int k = (int)(c % b.nk), j = (int)((c / b.nk) % b.nj), i = (int)(c / ((int64_t)b.nk * b.nj));
    if (i < ghost || j < ghost || k < ghost || i >= b.ni - ghost || j >= b.nj - ghost || k >= b.nk - ghost) continue;
    double pv[5];
    load_prim(b.q, b.N, c, gamma, pv);
    const bool ok = isfinite(pv[0]) && isfinite(pv[1]) && isfinite(pv[2]) && isfinite(pv[3]) && isfinite(pv[4]) &&
                    pv[0] > 0.0 && pv[4] > 0.0;
    bad += ok ? 0.0 : 1.0;
  }
  sbad[threadIdx.x] = bad;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sbad[threadIdx.x] += sbad[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sbad[0];
}

__global__ void __launch_bounds__(256) k_sum_parts(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double s[256];
  double a = 0.0;
  for (int t = threadIdx.x; t < n; t += blockDim.x) a += part[t];
  s[threadIdx.x] = a;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = s[0];
}

}  // namespace famrdp

// ===========================================================================
// Fused stage kernel: one launch per RK3 stage, every face flux and every
// viscous flux tensor computed once per tile.
//
// A workgroup owns a TI x TJ x TK tile (one thread per cell).
//  1. Stage primitives in LDS for the tile, a full one-cell halo box and a
//     second halo layer along each axis.  Halo cells are read at wrapped
//     (periodic) block coordinates: that is the reference's jnp.roll for the
//     viscous terms, and the inviscid faces never reach a wrapped cell (they
//     exist only between cells 1..n-2 of their axis).
//  2. Viscous flux tensor G (rhs/viscous.py:30-108) for the tile plus a
//     one-cell cross halo into LDS; every cell takes its viscous divergence.
//  3. For each axis, j, k, then i (the order the marching kernel sums them
//     in): MUSCL-2 + Roe face fluxes of the tile's low faces plus one layer
//     of high faces into an LDS face buffer (aliasing G), then
//     F(c+1/2) - F(c-1/2) for cells with 2 <= c_d <= n_d - 3
//     (rhs/invscd.py:100-131).
//  4. rhs = inv + vis and the Shu-Osher combination (solver/step.py:45-53).
// ===========================================================================
namespace famrdp {

// ---------------------------------------------------------------------------
// Inviscid faces of one axis D for a tile (rhs/invscd.py:53-131), shared by
// the fused and split stage kernels.  Faces of the tile: the low face of
// every cell (computed by the cell's own thread, with kxyz of the cell from
// registers) and the layer of high faces at the far end of the tile (dealt
// to the threads beyond the tile's cells, or after the low face when there
// are none).  Face fluxes go to the LDS buffer s_f (axes i, j: f * Pd + o,
// axis k: o * (TK + 1) + f, face f between local cells f-1 and f); after a
// barrier every cell with 2 <= c <= n-3 along D adds F(c+1/2) - F(c-1/2)
// (fluxes doubled, see roe_flux2) to A.  Ends with a barrier (s_f is reused by the next axis).
// ---------------------------------------------------------------------------
// kxyz[D, :] / 2 of the left neighbour of cell c along D (the left cell of the
// cell's own low face), loaded early so the face phase does not wait on it;
// zero where that face does not exist.
template <int D>
__device__ __forceinline__ void load_kl_own(const BlockDesc& b, int64_t c, int gl_d, bool own, double kl[3]) {
  const int64_t st = D == 0 ? (int64_t)b.nj * b.nk : (D == 1 ? (int64_t)b.nk : (int64_t)1);
  const bool ok = own && gl_d >= 1;
  const int64_t cl = ok ? c - st : c;   // always a valid address: a fixed number of loads
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double v = b.kxyz[(D * 3 + m) * b.N + cl];
    kl[m] = ok ? 0.5 * v : 0.0;
  }
}

template <int D, class T, int TI, int TJ, int TK, int NTH, int LIM>
__device__ __forceinline__ void face_axis(const BlockDesc& b, int i0, int j0, int k0, const double* s_pv,
                                          double* s_f, const double kkh[9], const double kl_own[3], bool own, int t,
                                          int x, int y, int z, const StageGas& gas, double A[5]) {
  EXACT_FP
  constexpr int NT = TI * TJ * TK;
  constexpr int Td = D == 0 ? TI : (D == 1 ? TJ : TK);
  constexpr int Pd = NT / Td;
  const int ni = b.ni, nj = b.nj, nk = b.nk;
  const int64_t N = b.N;
  const int64_t si = (int64_t)nj * nk, sj = nk;
  const int n_d = D == 0 ? ni : (D == 1 ? nj : nk);
  const int org_d = D == 0 ? i0 : (D == 1 ? j0 : k0);
  constexpr int64_t one = 1;
  const int64_t st_d = D == 0 ? si : (D == 1 ? sj : one);
  auto face = [&](int f, int lx, int ly, int lz, int slot, bool kr_own) {
    const int ai = i0 + lx, aj = j0 + ly, ak = k0 + lz;
    const int a = org_d + f - 1;          // cell left of the face (unwrapped)
    if (!(ai < ni && aj < nj && ak < nk && a >= 1 && a <= n_d - 3)) return;
    double p4[4][5];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const int sl = T::template axis_slot<D>(lx + (D == 0 ? s4 - 2 : 0), ly + (D == 1 ? s4 - 2 : 0),
                                              lz + (D == 2 ? s4 - 2 : 0));
#pragma unroll
      for (int v = 0; v < 5; ++v) p4[s4][v] = s_pv[v * T::NPVS + sl];
    }
    const int64_t cr = (int64_t)ai * si + (int64_t)aj * sj + ak;
    const int64_t cl = cr - st_d;    // a >= 1: in the block
    double kl[3], kr[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      kl[m] = kr_own ? kl_own[m] : 0.5 * b.kxyz[(D * 3 + m) * N + cl];
      kr[m] = kr_own ? kkh[D * 3 + m] : 0.5 * b.kxyz[(D * 3 + m) * N + cr];
    }
    double Fa[5];
    face_flux2<LIM>(p4[0], p4[1], p4[2], p4[3], kl, kr, gas, Fa);
#pragma unroll
    for (int v = 0; v < 5; ++v) s_f[v * T::NF + slot] = Fa[v];
  };
  const int loc_d = D == 0 ? x : (D == 1 ? y : z);
  const int o_own = D == 0 ? (y * TK + z) : (D == 1 ? (x * TK + z) : (x * TJ + y));
  if (t < NT) face(loc_d, x, y, z, D == 2 ? o_own * (TK + 1) + loc_d : loc_d * Pd + o_own, true);
  for (int h = (t >= NT ? t - NT : t + NTH - NT); h < Pd; h += NTH) {
    int lx, ly, lz;
    if constexpr (D == 0) { lx = TI; ly = h / TK; lz = h % TK; }
    else if constexpr (D == 1) { lx = h / TK; ly = TJ; lz = h % TK; }
    else { lx = h / TJ; ly = h % TJ; lz = TK; }
    face(Td, lx, ly, lz, D == 2 ? h * (TK + 1) + Td : Td * Pd + h, false);
  }
  __syncthreads();
  const int gl_d = D == 0 ? i0 + x : (D == 1 ? j0 + y : k0 + z);
  if (own && gl_d >= 2 && gl_d <= n_d - 3) {
    const int lo = D == 2 ? o_own * (TK + 1) + loc_d : loc_d * Pd + o_own;
    const int hi = D == 2 ? lo + 1 : lo + Pd;
#pragma unroll
    for (int v = 0; v < 5; ++v) A[v] = A[v] + (s_f[v * T::NF + hi] - s_f[v * T::NF + lo]);
  }
  __syncthreads();
}

template <int TI, int TJ, int TK, int W, bool ALL>
__device__ __forceinline__ void fused_cells_fill(const BlockDesc& b, int i0, int j0, int k0, int t,
                                                 FusedCells<TI, TJ, TK>& fc) {
  using C = FusedCells<TI, TJ, TK>;
  using T = typename C::T;
  const int ni = b.ni, nj = b.nj, nk = b.nk;
#pragma unroll
  for (int it = 0; it < C::NIT; ++it) {
    const int h = t + it * T::NT;
    const Loc3 l = T::pv_cell(h < T::NPV ? h : T::NPV - 1);
    fc.stage[it] = tile_cell_rel<W>(l.x + 2, l.y + 2, l.z + 2, i0, j0, k0, ni, nj, nk);
  }
  if constexpr (!ALL) return;
#pragma unroll
  for (int it = 1; it < C::NGIT; ++it) {
    const int h = t + it * T::NT;
    const Loc3 l = T::g_cell(h < T::NG ? h : T::NG - 1);
    fc.gh[it - 1] = tile_cell_rel<W>(l.x + 2, l.y + 2, l.z + 2, i0, j0, k0, ni, nj, nk);
  }
  const int x = t / (TJ * TK), y = (t / TK) % TJ, z = t % TK;
  fc.c = tile_cell<W>(i0 + x, j0 + y, k0 + z, ni, nj, nk);
}

// ALL = false: the staging slots only, for thread id t
template <int TI, int TJ, int TK, bool ALL = true>
__device__ __forceinline__ void fused_cells(const BlockDesc& b, int i0, int j0, int k0, int t,
                                            FusedCells<TI, TJ, TK>& fc) {
  const int w = fused_wrap_mode<TI, TJ, TK>(b.wrap_mod, i0, j0, k0, b.ni, b.nj, b.nk);
  if (w == WRAP_MOD) fused_cells_fill<TI, TJ, TK, WRAP_MOD, ALL>(b, i0, j0, k0, t, fc);
  else if (w == WRAP_NONE) fused_cells_fill<TI, TJ, TK, WRAP_NONE, ALL>(b, i0, j0, k0, t, fc);
  else fused_cells_fill<TI, TJ, TK, WRAP_ONCE, ALL>(b, i0, j0, k0, t, fc);
}

// v, hidden from the optimiser: values computed from it are computed again
// rather than kept in registers from an earlier, identical computation
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Staging loads of one tile into registers.  Every thread issues the same
// number of loads, so the compiler can wait for older loads without waiting
// for these.
template <int TI, int TJ, int TK>
__device__ __forceinline__ void fused_stage_loads(const BlockDesc& b, const double* __restrict__ qin,
                                                  const FusedCells<TI, TJ, TK>& fc, double qq[][5]) {
#pragma unroll
  for (int it = 0; it < FusedCells<TI, TJ, TK>::NIT; ++it) {
#pragma unroll
    for (int v = 0; v < 5; ++v) qq[it][v] = qin[v * b.N + fc.stage[it]];
  }
}

// One RK stage of one tile whose staging values are in qq (fused_stage_loads
// of this tile).  Global loads are grouped by the phase that first needs
// them: metrics of the G cells before the G phase, the faces' neighbour
// metrics and volume before the faces, the state at the update.
// RS (re-staging): the viscous tensors are kept in registers until every
// thread is done reading the primitives, then written over them; after the
// divergence the primitives are staged again (their loads issued before the
// divergence) for the faces.  Less LDS per workgroup, so more share a CU.
template <int TI, int TJ, int TK, int LIM, bool RS>
__device__ __forceinline__ void stage_tile_fused_regs(const BlockDesc& b, int i0, int j0, int k0,
                                                      const double* __restrict__ qin, const double* q0, double* qout,
                                                      const StageGas& gas, double dt, int stage,
                                                      const FusedCells<TI, TJ, TK>& fc, double qq[][5]) {
  EXACT_FP
  using T = FusedGeom<TI, TJ, TK>;
  constexpr int NIT = FusedCells<TI, TJ, TK>::NIT;
  __shared__ double lds[RS ? T::NLDS_RS : T::NLDS];
  double* s_pv = lds;                                  // [5][NPV]
  double* s_T = lds + 5 * T::NPV;                      // [NPV]   temperature of the staged cells
  double* s_g = RS ? lds : lds + 6 * T::NPV;           // [9][NG] (phase 2)
  double* s_f = RS ? lds + 5 * T::NPV : s_g;           // [5][NF] (phase 3)
  const int t = threadIdx.x;
  const int ni = b.ni, nj = b.nj, nk = b.nk;
  const int64_t N = b.N;
  const double cmu = uniform(gas.cmu * b.mu0);
  const StageCoef sc = stage_coef(stage, dt * b.dt_scale);
  const int x = t / (TJ * TK), y = (t / TK) % TJ, z = t % TK;
  const int gi = i0 + x, gj = j0 + y, gk = k0 + z;
  const bool own = gi < ni && gj < nj && gk < nk;
  // the tile cell of this thread (wrapped into the block when outside it)
  const int c = fc.c;

  // ---- 1. primitives from the staged registers --------------------------------
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int h = t + it * T::NT;
    if (h < T::NPV) {
      double pp[6];
      prim_and_temp(qq[it], gas, pp);
#pragma unroll
      for (int v = 0; v < 5; ++v) s_pv[v * T::NPV + h] = pp[v];
      s_T[h] = pp[5];
    }
  }

  // ---- metrics of the G cells --------------------------------------------------
  double kkh[9];   // kxyz / 2 of the thread's cell
#pragma unroll
  for (int m = 0; m < 9; ++m) kkh[m] = 0.5 * b.kxyz[m * N + c];
  constexpr int NGIT = FusedCells<TI, TJ, TK>::NGIT;
  double kh[NGIT > 1 ? NGIT - 1 : 1][9];
#pragma unroll
  for (int it = 1; it < NGIT; ++it) {
#pragma unroll
    for (int m = 0; m < 9; ++m) kh[it - 1][m] = 0.5 * b.kxyz[m * N + fc.gh[it - 1]];
  }
  __syncthreads();

  // ---- 2. viscous flux tensor and its divergence -----------------------------
  double gsave[RS ? NGIT : 1][9];
#pragma unroll
  for (int it = 0; it < NGIT; ++it) {
    const int h = t + it * T::NT;
    if (h >= T::NG) break;
    const Loc3 lc = T::g_cell(h);
    const int lx = lc.x, ly = lc.y, lz = lc.z;
    double kc[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) kc[m] = it == 0 ? kkh[m] : kh[it > 0 ? it - 1 : 0][m];
    double d[3][4];
    const int s0 = T::pv_slot(lx, ly, lz);
    const double uvwT[4] = {s_pv[T::NPV + s0], s_pv[2 * T::NPV + s0], s_pv[3 * T::NPV + s0], s_T[s0]};
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const int sp = T::pv_slot(lx + (l == 0), ly + (l == 1), lz + (l == 2));
      const int sm = T::pv_slot(lx - (l == 0), ly - (l == 1), lz - (l == 2));
      d[l][0] = s_pv[T::NPV + sp] - s_pv[T::NPV + sm];
      d[l][1] = s_pv[2 * T::NPV + sp] - s_pv[2 * T::NPV + sm];
      d[l][2] = s_pv[3 * T::NPV + sp] - s_pv[3 * T::NPV + sm];
      d[l][3] = s_T[sp] - s_T[sm];
    }
    double g9[9];
    viscous_flux_fast(uvwT, d, kc, cmu, gas, g9);
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      if constexpr (RS) gsave[it][m] = g9[m];
      else s_g[m * T::NG + h] = g9[m];
    }
  }
  __syncthreads();
  if constexpr (RS) {   // the primitives are no longer read: G goes over them
#pragma unroll
    for (int it = 0; it < NGIT; ++it) {
      const int h = t + it * T::NT;
      if (h < T::NG) {
#pragma unroll
        for (int m = 0; m < 9; ++m) s_g[m * T::NG + h] = gsave[it][m];
      }
    }
    // indices of the second staging computed again (held through the G
    // phase they would cost registers the three-per-CU budget lacks)
    FusedCells<TI, TJ, TK> fc2;
    fused_cells<TI, TJ, TK, false>(b, i0, j0, k0, opaque(t), fc2);
    fused_stage_loads<TI, TJ, TK>(b, qin, fc2, qq);
    __syncthreads();
  }
  double vis[4] = {0.0, 0.0, 0.0, 0.0};
  if (own) {
    const int sp[3] = {T::g_slot(x + 1, y, z), T::g_slot(x, y + 1, z), T::g_slot(x, y, z + 1)};
    const int sm[3] = {T::g_slot(x - 1, y, z), T::g_slot(x, y - 1, z), T::g_slot(x, y, z - 1)};
    double gm[9], gp[9], dj[9], dk[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      const double* Gc = s_g + m * T::NG;
      gm[m] = Gc[sm[0]];
      gp[m] = Gc[sp[0]];
      dj[m] = Gc[sp[1]] - Gc[sm[1]];
      dk[m] = Gc[sp[2]] - Gc[sm[2]];
    }
    visc_div_im(gm, kkh, vis);
    visc_div_jk(dj, dk, kkh, vis);
    visc_div_ip(gp, kkh, vis);
  }
  __syncthreads();   // G space is reused by the face buffer (and the primitives)
  if constexpr (RS) {
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int h = t + it * T::NT;
      if (h < T::NPV) {
        double pp[6];
        prim_and_temp(qq[it], gas, pp);
#pragma unroll
        for (int v = 0; v < 5; ++v) s_pv[v * T::NPV + h] = pp[v];
      }
    }
    __syncthreads();
  }

  // ---- 3. inviscid faces, axis by axis ---------------------------------------
  double kl0[3], kl1[3], kl2[3];
  load_kl_own<0>(b, c, gi, own, kl0);
  load_kl_own<1>(b, c, gj, own, kl1);
  load_kl_own<2>(b, c, gk, own, kl2);
  double A[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  const double rvh = own ? 0.5 * rcp(b.vol[c] + 1e-300) : 0.0;
  face_axis<1, T, TI, TJ, TK, T::NT, LIM>(b, i0, j0, k0, s_pv, s_f, kkh, kl1, own, t, x, y, z, gas, A);
  face_axis<2, T, TI, TJ, TK, T::NT, LIM>(b, i0, j0, k0, s_pv, s_f, kkh, kl2, own, t, x, y, z, gas, A);
  face_axis<0, T, TI, TJ, TK, T::NT, LIM>(b, i0, j0, k0, s_pv, s_f, kkh, kl0, own, t, x, y, z, gas, A);
  if (!own) return;

  // ---- 4. rhs and the RK3 combination ----------------------------------------
  double qs[5], qq0[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    qs[v] = qin[v * N + c];
    qq0[v] = stage == 1 ? 0.0 : q0[v * N + c];
  }
#pragma unroll
  for (int v = 0; v < 5; ++v) qout[v * N + c] = stage_update(sc, qq0[v], qs[v], A[v], rvh, v == 0 ? 0.0 : vis[v - 1]);
}

template <int TI, int TJ, int TK, int LIM, bool RS>
__device__ __forceinline__ void stage_tile_fused(const BlockDesc& b, int i0, int j0, int k0,
                                                 const double* __restrict__ qin, const double* q0, double* qout,
                                                 const StageGas& gas, double dt, int stage) {
  FusedCells<TI, TJ, TK> fc;
  fused_cells<TI, TJ, TK>(b, i0, j0, k0, (int)threadIdx.x, fc);
  double qq[FusedCells<TI, TJ, TK>::NIT][5];
  fused_stage_loads<TI, TJ, TK>(b, qin, fc, qq);
  stage_tile_fused_regs<TI, TJ, TK, LIM, RS>(b, i0, j0, k0, qin, q0, qout, gas, dt, stage, fc, qq);
}

// WPE: waves per SIMD the register allocation aims at (3 for the re-staging
// form at 256 threads: three workgroups per CU, at most 168 VGPRs).
template <int TI, int TJ, int TK, int LIM, bool RS, int WPE>
__global__ void __launch_bounds__(TI * TJ * TK) __attribute__((amdgpu_waves_per_eu(WPE)))
k_stage_fused(BlockDesc b, int stage, StageGas gas, double dt, int ntj, int ntk) {
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int tk = t % ntk, tj = (t / ntk) % ntj, ti = t / (ntk * ntj);
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  stage_tile_fused<TI, TJ, TK, LIM, RS>(b, ti * TI, tj * TJ, tk * TK, qin, b.q, qout, gas, dt, stage);
}

template <int TI, int TJ, int TK, int LIM, bool RS, int WPE>
__global__ void __launch_bounds__(TI * TJ * TK) __attribute__((amdgpu_waves_per_eu(WPE)))
k_stage_fused_batched(const BlockDesc* __restrict__ blocks, const Tile3* __restrict__ tiles, int stage, StageGas gas,
                      double dt) {
  const Tile3 tl = tiles[xcd_remap(blockIdx.x, gridDim.x)];
  const BlockDesc& b = blocks[tl.block];
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  stage_tile_fused<TI, TJ, TK, LIM, RS>(b, tl.i0, tl.j0, tl.k0, qin, b.q, qout, gas, dt, stage);
}

// ===========================================================================
// Split stage: two launches per RK3 stage (tile tables as the fused kernel).
//
//  k_visc_tensor  u, v, w, T of the tile and a one-cell cross halo staged in
//                 LDS; the viscous flux tensor G (rhs/viscous.py:30-108) of
//                 every cell, once, written to the plan's G buffer (9, N).
//  k_stage_split  primitives of the tile and a two-cell cross halo in LDS;
//                 divergence of G at the cell's six (wrapped) neighbours read
//                 from the G buffer; MUSCL-2 + Roe faces once per tile as in
//                 the fused kernel; the Shu-Osher combination.
// Every value is produced by the same expressions, on the same inputs, in
// the same order as in the fused kernel, so both kernels give the same bits;
// the split form holds no viscous tensor in LDS (43-74 KB per workgroup
// instead of 75-143 KB), so more workgroups share a CU.
// ===========================================================================
template <int TI, int TJ, int TK>
struct SplitGeom {
  static_assert(TI < WRAP_ONCE_MIN && TJ < WRAP_ONCE_MIN && TK < WRAP_ONCE_MIN, "tile longer than the single-wrap bound");
  static constexpr int NT = TI * TJ * TK;
  static constexpr int A0 = TJ * TK, A1 = TI * TK, A2 = TI * TJ;
  static constexpr int NP = NT + 4 * (A0 + A1 + A2);    // tile + two halo layers per side, per axis
  static constexpr int F0 = (TI + 1) * TJ * TK, F1 = TI * (TJ + 1) * TK, F2 = TI * TJ * (TK + 1);
  static constexpr int NF = F0 > F1 ? (F0 > F2 ? F0 : F2) : (F1 > F2 ? F1 : F2);
  static constexpr int NLDS = 5 * NP + 5 * NF;
  static constexpr int NPVS = NP;    // primitive slots (stride of a variable)

  // slot of the cell (lx, ly, lz) whose coordinate along D lies in
  // [-2, T_D + 1] and whose other two coordinates lie in the tile
  template <int D>
  __device__ static __forceinline__ int axis_slot(int lx, int ly, int lz) {
    if constexpr (D == 0) {
      const bool out = (unsigned)lx >= (unsigned)TI;
      return out ? NT + ((lx < 0 ? lx + 2 : lx - TI + 2) * TJ + ly) * TK + lz : (lx * TJ + ly) * TK + lz;
    } else if constexpr (D == 1) {
      const bool out = (unsigned)ly >= (unsigned)TJ;
      return out ? NT + 4 * A0 + ((ly < 0 ? ly + 2 : ly - TJ + 2) * TI + lx) * TK + lz : (lx * TJ + ly) * TK + lz;
    } else {
      const bool out = (unsigned)lz >= (unsigned)TK;
      return out ? NT + 4 * (A0 + A1) + ((lz < 0 ? lz + 2 : lz - TK + 2) * TI + lx) * TJ + ly
                 : (lx * TJ + ly) * TK + lz;
    }
  }
  // threads that give every axis's faces one pass (a multiple of 64)
  static constexpr int NTH1 = (NF + 63) / 64 * 64;

  // slot of a cell that lies in the tile or on the halo layers of one axis
  // (written with selects only: no divergent branches in the face loops)
  __device__ static __forceinline__ int p_slot(int x, int y, int z) {
    const bool ox = (unsigned)x >= (unsigned)TI, oy = (unsigned)y >= (unsigned)TJ, oz = (unsigned)z >= (unsigned)TK;
    const int lx = x < 0 ? x + 2 : x - TI + 2, ly = y < 0 ? y + 2 : y - TJ + 2, lz = z < 0 ? z + 2 : z - TK + 2;
    const int s_in = (x * TJ + y) * TK + z;
    const int s_x = NT + (lx * TJ + y) * TK + z;
    const int s_y = NT + 4 * A0 + (ly * TI + x) * TK + z;
    const int s_z = NT + 4 * (A0 + A1) + (lz * TI + x) * TJ + y;
    return ox ? s_x : (oy ? s_y : (oz ? s_z : s_in));
  }
  // inverse of p_slot
  __device__ static __forceinline__ int3 p_cell(int h) {
    if (h < NT) return make_int3(h / (TJ * TK), (h / TK) % TJ, h % TK);
    h -= NT;
    if (h < 4 * A0) {
      const int l = h / A0, r = h % A0;
      return make_int3(l < 2 ? l - 2 : TI + l - 2, r / TK, r % TK);
    }
    h -= 4 * A0;
    if (h < 4 * A1) {
      const int l = h / A1, r = h % A1;
      return make_int3(r / TK, l < 2 ? l - 2 : TJ + l - 2, r % TK);
    }
    h -= 4 * A1;
    const int l = h / A2, r = h % A2;
    return make_int3(r / TJ, r % TJ, l < 2 ? l - 2 : TK + l - 2);
  }
};

template <int TI, int TJ, int TK>
__device__ __forceinline__ void visc_tile(const BlockDesc& b, int i0, int j0, int k0, const double* __restrict__ qin,
                                          const StageGas& gas) {
  EXACT_FP
  using T = FusedGeom<TI, TJ, TK>;       // g_slot / g_cell: tile + one-cell cross halo
  __shared__ double s_w[4 * T::NG];      // u, v, w, T
  const int t = threadIdx.x;
  const int ni = b.ni, nj = b.nj, nk = b.nk;
  const int64_t N = b.N;
  const int64_t si = (int64_t)nj * nk, sj = nk;
  const double cmu = uniform(gas.cmu * b.mu0);
  {
    constexpr int NIT = (T::NG + T::NT - 1) / T::NT;
    int cc[NIT];
    auto cells = [&](auto mod) {
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int h = t + it * T::NT;
        const Loc3 lc = T::g_cell(h < T::NG ? h : T::NG - 1);
        cc[it] = tile_cell<decltype(mod)::value>(i0 + lc.x, j0 + lc.y, k0 + lc.z, ni, nj, nk);
      }
    };
    if (b.wrap_mod) cells(std::true_type{});
    else cells(std::false_type{});
    double qq[NIT][5];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int h = t + it * T::NT;
      if (h < T::NG) {
#pragma unroll
        for (int v = 0; v < 5; ++v) qq[it][v] = qin[v * N + cc[it]];
      }
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int h = t + it * T::NT;
      if (h < T::NG) {
        double pp[6];
        prim_and_temp(qq[it], gas, pp);
        s_w[h] = pp[1];
        s_w[T::NG + h] = pp[2];
        s_w[2 * T::NG + h] = pp[3];
        s_w[3 * T::NG + h] = pp[5];
      }
    }
  }
  __syncthreads();
  const int x = t / (TJ * TK), y = (t / TK) % TJ, z = t % TK;
  const int gi = i0 + x, gj = j0 + y, gk = k0 + z;
  if (gi >= ni || gj >= nj || gk >= nk) return;
  const int64_t c = (int64_t)gi * si + (int64_t)gj * sj + gk;
  const int s0 = T::g_slot(x, y, z);
  const double uvwT[4] = {s_w[s0], s_w[T::NG + s0], s_w[2 * T::NG + s0], s_w[3 * T::NG + s0]};
  double d[3][4];
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const int sp = T::g_slot(x + (l == 0), y + (l == 1), z + (l == 2));
    const int sm = T::g_slot(x - (l == 0), y - (l == 1), z - (l == 2));
#pragma unroll
    for (int v = 0; v < 4; ++v) d[l][v] = s_w[v * T::NG + sp] - s_w[v * T::NG + sm];
  }
  double kc[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) kc[m] = 0.5 * b.kxyz[m * N + c];
  double g9[9];
  viscous_flux_fast(uvwT, d, kc, cmu, gas, g9);
#pragma unroll
  for (int m = 0; m < 9; ++m) b.G[m * N + c] = g9[m];
}

template <int TI, int TJ, int TK, int NTH, int LIM>
__device__ __forceinline__ void stage_tile_split(const BlockDesc& b, int i0, int j0, int k0,
                                                 const double* __restrict__ qin, const double* q0, double* qout,
                                                 const StageGas& gas, double dt, int stage) {
  EXACT_FP
  using T = SplitGeom<TI, TJ, TK>;
  static_assert(NTH >= T::NT && NTH % 64 == 0, "stage kernel needs a thread per cell");
  __shared__ double lds[T::NLDS];
  double* s_pv = lds;                    // [5][NP]
  double* s_f = lds + 5 * T::NP;         // [5][NF]
  const int t = threadIdx.x;
  const int ni = b.ni, nj = b.nj, nk = b.nk;
  const int64_t N = b.N;
  const int64_t si = (int64_t)nj * nk, sj = nk;
  const StageCoef sc = stage_coef(stage, dt * b.dt_scale);
  // threads t < NT own cell (x, y, z) of the tile; all NTH threads compute faces
  const int x = t / (TJ * TK), y = (t / TK) % TJ, z = t % TK;
  const int gi = i0 + x, gj = j0 + y, gk = k0 + z;
  const bool own = t < T::NT && gi < ni && gj < nj && gk < nk;
  // the thread's cell (wrapped into the block when outside it: a valid
  // address) and its staging cells
  constexpr int NIT = (T::NP + NTH - 1) / NTH;
  int c, cc[NIT];
  auto cells = [&](auto mod) {
    constexpr bool M = decltype(mod)::value;
    c = tile_cell<M>(gi, gj, gk, ni, nj, nk);
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int h = t + it * NTH;
      const int3 lc = T::p_cell(h < T::NP ? h : T::NP - 1);
      cc[it] = tile_cell<M>(i0 + lc.x, j0 + lc.y, k0 + lc.z, ni, nj, nk);
    }
  };
  if (b.wrap_mod) cells(std::true_type{});
  else cells(std::false_type{});

  // ---- 1. primitives of the tile and the two-cell cross halo ------------------
  {
    double qq[NIT][5];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int h = t + it * NTH;
      if (h < T::NP) {
#pragma unroll
        for (int v = 0; v < 5; ++v) qq[it][v] = qin[v * N + cc[it]];
      }
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int h = t + it * NTH;
      if (h < T::NP) {
        double pp[6];
        prim_and_temp(qq[it], gas, pp);
#pragma unroll
        for (int v = 0; v < 5; ++v) s_pv[v * T::NP + h] = pp[v];
      }
    }
  }

  // ---- 2. divergence of the viscous tensor (G of the six wrapped neighbours) ---
  double kkh[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) kkh[m] = own ? 0.5 * b.kxyz[m * N + c] : 0.0;
  double kl0[3], kl1[3], kl2[3];
  load_kl_own<0>(b, c, gi, own, kl0);
  load_kl_own<1>(b, c, gj, own, kl1);
  load_kl_own<2>(b, c, gk, own, kl2);
  double vis[4] = {0.0, 0.0, 0.0, 0.0};
  if (own) {
    const int64_t cp[3] = {c + (int64_t)(wrap_p(gi, ni) - gi) * si, c + (int64_t)(wrap_p(gj, nj) - gj) * sj,
                           c + (wrap_p(gk, nk) - gk)};
    const int64_t cm[3] = {c + (int64_t)(wrap_m(gi, ni) - gi) * si, c + (int64_t)(wrap_m(gj, nj) - gj) * sj,
                           c + (wrap_m(gk, nk) - gk)};
    double gm[9], gp[9], dj[9], dk[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      const double* __restrict__ Gc = b.G + m * N;
      gm[m] = Gc[cm[0]];
      gp[m] = Gc[cp[0]];
      dj[m] = Gc[cp[1]] - Gc[cm[1]];
      dk[m] = Gc[cp[2]] - Gc[cm[2]];
    }
    visc_div_im(gm, kkh, vis);
    visc_div_jk(dj, dk, kkh, vis);
    visc_div_ip(gp, kkh, vis);
  }
  __syncthreads();

  // ---- 3. inviscid faces, axis by axis ---------------------------------------
  double A[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  const double rvh = own ? 0.5 * rcp(b.vol[c] + 1e-300) : 0.0;
  face_axis<1, T, TI, TJ, TK, NTH, LIM>(b, i0, j0, k0, s_pv, s_f, kkh, kl1, own, t, x, y, z, gas, A);
  face_axis<2, T, TI, TJ, TK, NTH, LIM>(b, i0, j0, k0, s_pv, s_f, kkh, kl2, own, t, x, y, z, gas, A);
  face_axis<0, T, TI, TJ, TK, NTH, LIM>(b, i0, j0, k0, s_pv, s_f, kkh, kl0, own, t, x, y, z, gas, A);
  if (!own) return;

  // ---- 4. rhs and the RK3 combination ----------------------------------------
  double qs[5], qq0[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    qs[v] = qin[v * N + c];
    qq0[v] = stage == 1 ? 0.0 : q0[v * N + c];
  }
#pragma unroll
  for (int v = 0; v < 5; ++v) qout[v * N + c] = stage_update(sc, qq0[v], qs[v], A[v], rvh, v == 0 ? 0.0 : vis[v - 1]);
}

template <int TI, int TJ, int TK>
__global__ void __launch_bounds__(TI * TJ * TK) k_visc_tensor(BlockDesc b, int stage, StageGas gas, int ntj, int ntk) {
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int tk = t % ntk, tj = (t / ntk) % ntj, ti = t / (ntk * ntj);
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  visc_tile<TI, TJ, TK>(b, ti * TI, tj * TJ, tk * TK, qin, gas);
}

template <int TI, int TJ, int TK, int NTH, int LIM>
__global__ void __launch_bounds__(NTH) k_stage_split(BlockDesc b, int stage, StageGas gas, double dt, int ntj, int ntk) {
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int tk = t % ntk, tj = (t / ntk) % ntj, ti = t / (ntk * ntj);
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  stage_tile_split<TI, TJ, TK, NTH, LIM>(b, ti * TI, tj * TJ, tk * TK, qin, b.q, qout, gas, dt, stage);
}

template <int TI, int TJ, int TK>
__global__ void __launch_bounds__(TI * TJ * TK) k_visc_tensor_batched(const BlockDesc* __restrict__ blocks,
                                                                      const Tile3* __restrict__ tiles, int stage,
                                                                      StageGas gas) {
  const Tile3 tl = tiles[xcd_remap(blockIdx.x, gridDim.x)];
  const BlockDesc& b = blocks[tl.block];
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  visc_tile<TI, TJ, TK>(b, tl.i0, tl.j0, tl.k0, qin, gas);
}

template <int TI, int TJ, int TK, int NTH, int LIM>
__global__ void __launch_bounds__(NTH) k_stage_split_batched(const BlockDesc* __restrict__ blocks,
                                                             const Tile3* __restrict__ tiles, int stage, StageGas gas,
                                                             double dt) {
  const Tile3 tl = tiles[xcd_remap(blockIdx.x, gridDim.x)];
  const BlockDesc& b = blocks[tl.block];
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  stage_tile_split<TI, TJ, TK, NTH, LIM>(b, tl.i0, tl.j0, tl.k0, qin, b.q, qout, gas, dt, stage);
}

}  // namespace famrdp

#include "famrdp_march.h"
#include "famrdp_wide.h"
#include "famrdp_rhs.h"

namespace famrdp {

// Stage-kernel variants the autotuner chooses from (ids 0-4 and 10-13
// fused, 5-9 split pair, 14- i-marching).  Fused kernel: (id, TI, TJ, TK, re-staging, waves
// per SIMD for the register allocation), one thread per cell.  Split pair:
// (id, TI, TJ, TK, threads of the stage kernel): with one thread per cell an
// axis's faces take two passes, with a thread per face (NTH1) one.
#define FAMRDP_TILE_VARIANTS(X) \
  X(0, 8, 4, 8, false, 1)       \
  X(1, 4, 8, 16, false, 1)      \
  X(2, 8, 4, 16, false, 1)      \
  X(3, 4, 8, 8, false, 1)       \
  X(4, 4, 8, 8, true, 3)        \
  X(10, 8, 4, 8, true, 3)       \
  X(11, 8, 8, 4, true, 3)       \
  X(12, 4, 4, 16, true, 3)      \
  X(13, 8, 8, 8, true, 4)
#define FAMRDP_SPLIT_VARIANTS(X)  \
  X(5, 4, 4, 16, 256)             \
  X(6, 4, 8, 8, 256)              \
  X(7, 8, 8, 8, 512)              \
  X(8, 2, 8, 16, 256)             \
  X(9, 4, 8, 8, 320)
// i-marching kernel: (id, TJ, TK, segment length L about which march_len
// chooses, waves per SIMD); its tile table holds (2 x segment index + strip bit, j0, k0) per march_tiling.
// The 10-plane segments of 18 are for blocks of about 100^3 cells, which the
// longer segments leave with fewer workgroups than the GPU holds at once.
#define FAMRDP_MARCH_VARIANTS(X) \
  X(14, 16, 16, 32, 2)           \
  X(15, 8, 32, 20, 2)            \
  X(16, 8, 32, 32, 2)            \
  X(17, 8, 32, 52, 2)            \
  X(18, 8, 32, 10, 2)
// Wide kernel (famrdp_wide.h): (id, TI, TJ, TK).
#define FAMRDP_WIDE_VARIANTS(X) \
  X(19, 3, 4, 4)                \
  X(20, 4, 4, 8)
constexpr int NUM_TILE_VARIANTS = 21;

inline bool is_march_variant(int v) {
  switch (v) {
#define FAMRDP_IM(id, b, c, l, w) case id: return true;
    FAMRDP_MARCH_VARIANTS(FAMRDP_IM)
#undef FAMRDP_IM
    default: return false;
  }
}

inline bool is_wide_variant(int v) {
  switch (v) {
#define FAMRDP_IW(id, a, b, c) case id: return true;
    FAMRDP_WIDE_VARIANTS(FAMRDP_IW)
#undef FAMRDP_IW
    default: return false;
  }
}

inline void tile_dims(int v, int& ti, int& tj, int& tk) {
  switch (v) {
#define FAMRDP_TD5(id, a, b, c, n) case id: ti = a; tj = b; tk = c; return;
#define FAMRDP_TD6(id, a, b, c, rs, w) case id: ti = a; tj = b; tk = c; return;
#define FAMRDP_TDM(id, b, c, l, w) case id: ti = l; tj = b; tk = c; return;
#define FAMRDP_TDW(id, a, b, c) case id: ti = a; tj = b; tk = c; return;
    FAMRDP_TILE_VARIANTS(FAMRDP_TD6)
    FAMRDP_SPLIT_VARIANTS(FAMRDP_TD5)
    FAMRDP_MARCH_VARIANTS(FAMRDP_TDM)
    FAMRDP_WIDE_VARIANTS(FAMRDP_TDW)
#undef FAMRDP_TDW
#undef FAMRDP_TD5
#undef FAMRDP_TD6
#undef FAMRDP_TDM
    default: ti = 4; tj = 4; tk = 16;
  }
}

// Planes a workgroup of variant v takes along i when these blocks are launched
// together: a tile's, or at most a segment's.
inline int variant_len(int v, int nblocks, const int32_t* dims, int ncu) {
  int TI, TJ, TK;
  tile_dims(v, TI, TJ, TK);
  return is_march_variant(v) ? march_len(TJ, TK, TI, nblocks, dims, 2 * ncu) : TI;
}

// Tiles of one block with variant v (not a marching one).
inline int64_t stage_tiles(int v, int ni, int nj, int nk) {
  int TI, TJ, TK;
  tile_dims(v, TI, TJ, TK);
  return (int64_t)((ni + TI - 1) / TI) * ((nj + TJ - 1) / TJ) * ((nk + TK - 1) / TK);
}

// The variant of blocks that were not tuned: of the five below the one whose
// stage should be shortest.  A stage lasts as its workgroups per compute unit
// (n, rounded up) take; measured (minmod; van Leer is 10-17 % longer for all
// alike), in us, for cubes of 12^3 to 124^3 cells, flat and long blocks and
// lattices of small ones, the lines hold within 10 %:
//   19 wide 3x4x4    3.5 + 1.75 n   (20^3 5.4, 36^3 9.9, 72^3 54.8)
//   20 wide 4x4x8    1.5 + 5.6 n    (32^3 7.6, 44^3 17.2)
//    1 fused 4x8x16  15.3 n         (44^3 15.8, 60^3 30.7, 72^3 58.6)
//   12 re-staging    5 + 6.5 n      (52^3 24.2, 84^3 75.2, 104^3 125.2)
//   18 marching      6.9 per plane of march_len's count, 4.7 with no more than
//                    a workgroup per CU (72^3 50.5, 96^3 66.2, 112^3 111, 124^3 151)
// The fused kernel of 8x4x8 cells that every untuned block took before:
// 12.1 at 20^3, 27.5 at 52^3, 65.8 at 80^3, 109 at 96^3, 258 at 124^3.
inline int default_variant(int nblocks, const int32_t* dims, int ncu, bool fits32) {
  struct Line { int v; double base, per; };
  constexpr Line lines[] = {{19, 3.5, 1.75}, {20, 1.5, 5.6}, {1, 0, 15.3}, {12, 5, 6.5}, {18, 0, 6.9}};
  int best = 12;
  double best_t = 1e300;
  for (const Line& l : lines) {
    if (!fits32 && (is_march_variant(l.v) || is_wide_variant(l.v))) continue;
    double t;
    if (is_march_variant(l.v)) {
      int TI, TJ, TK;
      int64_t n = 0;
      tile_dims(l.v, TI, TJ, TK);
      march_len(TJ, TK, TI, nblocks, dims, 2 * ncu, &t, &n);
      t *= n <= ncu ? 4.7 : l.per;
    } else {
      int64_t n = 0;
      for (int b = 0; b < nblocks; ++b) n += stage_tiles(l.v, dims[3 * b], dims[3 * b + 1], dims[3 * b + 2]);
      t = l.base + l.per * (double)((n + ncu - 1) / ncu);
    }
    if (t < best_t) { best_t = t; best = l.v; }
  }
  return best;
}

// One stage of one block (plain launch) with variant v; the limiter is a
// template parameter of the stage kernels (LIM_MINMOD / LIM_VANLEER).
template <int LIM>
inline void launch_stage_lim(int v, const BlockDesc& d, int stage, const StageGas& gas, double dt, int ncu,
                             hipStream_t st) {
  int TI, TJ, TK;
  tile_dims(v, TI, TJ, TK);
  const int nti = (d.ni + TI - 1) / TI, ntj = (d.nj + TJ - 1) / TJ, ntk = (d.nk + TK - 1) / TK;
  const int nt = nti * ntj * ntk;
  switch (v) {
#define FAMRDP_TL(id, a, b, c, rs, w) \
  case id: k_stage_fused<a, b, c, LIM, rs, w><<<nt, a * b * c, 0, st>>>(d, stage, gas, dt, ntj, ntk); return;
    FAMRDP_TILE_VARIANTS(FAMRDP_TL)
#undef FAMRDP_TL
#define FAMRDP_SL(id, a, b, c, n)                                                       \
  case id:                                                                              \
    k_visc_tensor<a, b, c><<<nt, a * b * c, 0, st>>>(d, stage, gas, ntj, ntk);          \
    k_stage_split<a, b, c, n, LIM><<<nt, n, 0, st>>>(d, stage, gas, dt, ntj, ntk);      \
    return;
    FAMRDP_SPLIT_VARIANTS(FAMRDP_SL)
#undef FAMRDP_SL
#define FAMRDP_ML(id, b, c, l, w)                                                                          \
  case id: {                                                                                               \
    const int32_t dims[3] = {d.ni, d.nj, d.nk};                                                            \
    const int len = variant_len(v, 1, dims, ncu);                                                          \
    const int nwg = march_nseg(d.ni, len) * march_tiling(b, c, d.nj, d.nk).count();                        \
    k_stage_march<b, c, LIM, w><<<nwg, b * c, 0, st>>>(d, stage, gas, dt, len);                            \
    return;                                                                                                \
  }
    FAMRDP_MARCH_VARIANTS(FAMRDP_ML)
#undef FAMRDP_ML
#define FAMRDP_WL(id, a, b, c) \
  case id: k_stage_wide<a, b, c, LIM><<<nt, WideGeom<a, b, c>::NTH, 0, st>>>(d, stage, gas, dt, ntj, ntk); return;
    FAMRDP_WIDE_VARIANTS(FAMRDP_WL)
#undef FAMRDP_WL
  }
}

inline StageGas stage_gas(const Gas& g) {
  const double gm1 = g.gamma - 1.0;
  return StageGas{gm1, 0.5 * gm1, 2.0 * g.gamma / gm1, g.R, 1.0 / g.R, g.Ts, (g.T0 + g.Ts) / (g.T0 * std::sqrt(g.T0)),
                  g.gamma * g.R / (gm1 * g.Pr_lam)};
}

inline void launch_fused(int v, const BlockDesc& d, int stage, const Gas& gas, int lim, double dt, int ncu,
                         hipStream_t st) {
  const StageGas sg = stage_gas(gas);
  if (lim == LIM_VANLEER) launch_stage_lim<LIM_VANLEER>(v, d, stage, sg, dt, ncu, st);
  else launch_stage_lim<LIM_MINMOD>(v, d, stage, sg, dt, ncu, st);
}

// One stage of every block in one launch (two for the split pair) over a tile
// table built for v (len: variant_len of all of them).
template <int LIM>
inline void launch_stage_batched_lim(int v, const BlockDesc* blocks, const Tile3* tiles, int ntiles, int stage,
                                     const StageGas& gas, double dt, int len, hipStream_t st) {
  switch (v) {
#define FAMRDP_TB(id, a, b, c, rs, w)                                                                       \
  case id:                                                                                                   \
    k_stage_fused_batched<a, b, c, LIM, rs, w><<<ntiles, a * b * c, 0, st>>>(blocks, tiles, stage, gas, dt); \
    return;
    FAMRDP_TILE_VARIANTS(FAMRDP_TB)
#undef FAMRDP_TB
#define FAMRDP_SB(id, a, b, c, n)                                                                  \
  case id:                                                                                         \
    k_visc_tensor_batched<a, b, c><<<ntiles, a * b * c, 0, st>>>(blocks, tiles, stage, gas);       \
    k_stage_split_batched<a, b, c, n, LIM><<<ntiles, n, 0, st>>>(blocks, tiles, stage, gas, dt);   \
    return;
    FAMRDP_SPLIT_VARIANTS(FAMRDP_SB)
#undef FAMRDP_SB
#define FAMRDP_MB(id, b, c, l, w)                                                                        \
  case id:                                                                                                \
    k_stage_march_batched<b, c, LIM, w><<<ntiles, b * c, 0, st>>>(blocks, tiles, stage, gas, dt, len);    \
    return;
    FAMRDP_MARCH_VARIANTS(FAMRDP_MB)
#undef FAMRDP_MB
#define FAMRDP_WB(id, a, b, c)                                                                                      \
  case id:                                                                                                          \
    k_stage_wide_batched<a, b, c, LIM><<<ntiles, WideGeom<a, b, c>::NTH, 0, st>>>(blocks, tiles, stage, gas, dt);   \
    return;
    FAMRDP_WIDE_VARIANTS(FAMRDP_WB)
#undef FAMRDP_WB
  }
}

inline void launch_fused_batched(int v, const BlockDesc* blocks, const Tile3* tiles, int ntiles, int stage,
                                 const Gas& gas, int lim, double dt, int len, hipStream_t st) {
  const StageGas sg = stage_gas(gas);
  if (lim == LIM_VANLEER) launch_stage_batched_lim<LIM_VANLEER>(v, blocks, tiles, ntiles, stage, sg, dt, len, st);
  else launch_stage_batched_lim<LIM_MINMOD>(v, blocks, tiles, ntiles, stage, sg, dt, len, st);
}

}  // namespace famrdp

// Pointwise FP64 numerics of famrdp_jax's RHS path, shared by every kernel.
//
// Each function restates one reference formula in the reference's evaluation
// order (so results track the CPU restatement to rounding), written as plain
// scalar FP64 code for one cell or one face.  Citations are to the reference
// repository (famrdp_jax/...).
#pragma once

#include <hip/hip_runtime.h>

#define FD __host__ __device__ __forceinline__

namespace famrdp {

enum Limiter : int { LIM_MINMOD = 0, LIM_VANLEER = 1 };

// NaN semantics.  jnp.maximum / jnp.minimum / jnp.sign return NaN when an
// operand is NaN, while C's fmax / fmin return the other operand; the floors
// and the limiter below use these selects so a NaN state goes NaN the way
// the reference's does.
//   max_floor(x, c) = jnp.maximum(x, c) for a constant floor c (NaN x -> NaN)
FD double max_floor(double x, double c) { return x < c ? c : x; }
//   jnp.minimum(a, b) / jnp.maximum(a, b)
FD double min_nan(double a, double b) { return a != a ? a : (b != b ? b : fmin(a, b)); }
FD double max_nan(double a, double b) { return a != a ? a : (b != b ? b : fmax(a, b)); }

// physics/eos.py:12-17
FD void cons_to_prim(const double q[5], double g, double pv[5]) {
  const double rho = q[0];
  const double u = q[1] / rho, v = q[2] / rho, w = q[3] / rho;
  const double ke = 0.5 * (u * u + v * v + w * w);
  pv[0] = rho; pv[1] = u; pv[2] = v; pv[3] = w;
  pv[4] = (g - 1.0) * (q[4] - rho * ke);
}

// physics/eos.py:5-9
FD void prim_to_cons(const double pv[5], double g, double U[5]) {
  const double rho = pv[0], u = pv[1], v = pv[2], w = pv[3], p = pv[4];
  const double ke = 0.5 * (u * u + v * v + w * w);
  U[0] = rho; U[1] = rho * u; U[2] = rho * v; U[3] = rho * w;
  U[4] = p / (g - 1.0) + rho * ke;
}

// physics/eos.py:24-25; (T/T0)**1.5 evaluated as x*sqrt(x) (NaN for T < 0,
// as the reference's power)
FD double sutherland(double T, double mu0, double T0, double Ts) {
  const double x = T / T0;
  return mu0 * (x * sqrt(x)) * (T0 + Ts) / (T + Ts);
}

// jnp.sign: -1, 0 (signed), +1, NaN for NaN
FD double sgn(double a) { return a > 0.0 ? 1.0 : (a < 0.0 ? -1.0 : a); }

// physics/reconstruct/muscl2.py:5-7: s = sign(a)*max(sign(a)sign(b),0); s*min(|a|,|b|)
// (NaN in either argument gives NaN)
FD double minmod(double a, double b) {
  const double sa = sgn(a);
  const double s = sa * max_nan(sa * sgn(b), 0.0);
  return s * min_nan(fabs(a), fabs(b));
}

// physics/reconstruct/muscl2.py:10-12
FD double vanleer(double a, double b) {
  const double ab = a + b;
  const double safe = fabs(ab) > 1e-30 ? ab : 1.0;
  return (a * b > 0.0) ? (2.0 * a * b / safe) : 0.0;
}

FD double limit(int lim, double a, double b) {
  return lim == LIM_VANLEER ? vanleer(a, b) : minmod(a, b);
}

// minmod without the sign products: same-sign arguments give the smaller
// magnitude with a's sign, anything else gives zero (the reference's
// s * min(|a|,|b|) with s in {-1, 0, 1}; a zero's sign never reaches q).
// As the median of (a, b, 0), max(min(a,b), min(max(a,b),0)): both positive
// gives max(min(a,b), 0) = min(a,b), both negative max(min(a,b), max(a,b)) =
// max(a,b) (the one nearer zero), mixed signs or a zero give 0 -- the
// reference's value exactly, in four min/max, for non-NaN arguments.  A NaN
// argument is dropped here (hardware min/max return the other operand; two
// NaNs give 0); the face states that use it restore the reference's NaN
// propagation for the whole four-cell stencil instead, at two instructions
// per face rather than two per limiter call.
FD double minmod_fast(double a, double b) { return fmax(fmin(a, b), fmin(fmax(a, b), 0.0)); }

// The same value as a clamped to the interval between 0 and b (b > 0: a in
// [0, b]; b < 0: a in [b, 0]): the interval, two min/max, serves both slopes
// of a face, whose cells share the difference b.
FD void minmod_range(double b, double& lo, double& hi) { lo = fmin(b, 0.0); hi = fmax(b, 0.0); }
FD double minmod_in(double a, double lo, double hi) { return fmin(fmax(a, lo), hi); }

// flux/roe.py:5-18
FD void physical_flux(const double U[5], const double n[3], double g, double F[5]) {
  const double rho = max_floor(U[0], 1e-300);
  const double u = U[1] / rho, v = U[2] / rho, w = U[3] / rho;
  const double ke = 0.5 * (u * u + v * v + w * w);
  const double p = (g - 1.0) * (U[4] - rho * ke);
  const double un = u * n[0] + v * n[1] + w * n[2];
  const double H = (U[4] + p) / rho;
  F[0] = rho * un;
  F[1] = rho * u * un + p * n[0];
  F[2] = rho * v * un + p * n[1];
  F[3] = rho * w * un + p * n[2];
  F[4] = rho * H * un;
}

// flux/roe.py:21-85: Roe flux for a unit normal n, Harten fix on lambda1/5.
// fence(x, ...) marks values as computed by then; a kernel that is short of
// registers passes one that holds the compiler to it.
struct NoFence {
  template <class... T>
  FD void operator()(T&...) const {}
};
template <class Fence = NoFence>
FD void roe_flux(const double UL[5], const double UR[5], const double n[3], double g,
                 double eps_entropy, double F[5], Fence fence = Fence{}) {
  const double rhoL = max_floor(UL[0], 1e-300), rhoR = max_floor(UR[0], 1e-300);
  double uL = UL[1] / rhoL, vL = UL[2] / rhoL, wL = UL[3] / rhoL;
  fence(uL, vL, wL);
  double uR = UR[1] / rhoR, vR = UR[2] / rhoR, wR = UR[3] / rhoR;
  fence(uR, vR, wR);
  const double keL = 0.5 * (uL * uL + vL * vL + wL * wL);
  const double keR = 0.5 * (uR * uR + vR * vR + wR * wR);
  const double pL = (g - 1.0) * (UL[4] - rhoL * keL);
  const double pR = (g - 1.0) * (UR[4] - rhoR * keR);
  double HL = (UL[4] + pL) / rhoL;
  fence(HL);
  double HR = (UR[4] + pR) / rhoR;
  fence(HR);

  const double sqL = sqrt(rhoL), sqR = sqrt(rhoR);
  const double ss = max_floor(sqL + sqR, 1e-150);
  double uh = (sqL * uL + sqR * uR) / ss;
  fence(uh);
  double vh = (sqL * vL + sqR * vR) / ss;
  fence(vh);
  double wh = (sqL * wL + sqR * wR) / ss;
  fence(wh);
  double Hh = (sqL * HL + sqR * HR) / ss;
  fence(Hh);
  const double q2 = uh * uh + vh * vh + wh * wh;
  double c2 = max_floor((g - 1.0) * (Hh - 0.5 * q2), 1e-30);
  double ch = sqrt(c2);
  double unh = uh * n[0] + vh * n[1] + wh * n[2];
  double rhoh = sqL * sqR;
  fence(c2, ch, unh, rhoh);

  const double eps = eps_entropy * (fabs(unh) + ch);
  const double lam1 = unh - ch, lam5 = unh + ch;
  double al1 = fabs(lam1) >= eps ? fabs(lam1) : 0.5 * (lam1 * lam1 / eps + eps);
  fence(al1);
  double al5 = fabs(lam5) >= eps ? fabs(lam5) : 0.5 * (lam5 * lam5 / eps + eps);
  fence(al5);
  const double al2 = fabs(unh);

  double dU[5];
  for (int v = 0; v < 5; ++v) dU[v] = UR[v] - UL[v];
  const double dp = (g - 1.0) * (dU[4] - uh * dU[1] - vh * dU[2] - wh * dU[3] + 0.5 * q2 * dU[0]);
  const double dun = (dU[1] * n[0] + dU[2] * n[1] + dU[3] * n[2]) - unh * dU[0];
  double a1 = (dp - rhoh * ch * dun) / (2.0 * c2);
  fence(a1);
  double a5 = (dp + rhoh * ch * dun) / (2.0 * c2);
  fence(a5);
  double a23 = dU[0] - dp / c2;
  fence(a23);

  const double R1[5] = {1.0, uh - ch * n[0], vh - ch * n[1], wh - ch * n[2], Hh - ch * unh};
  const double R5[5] = {1.0, uh + ch * n[0], vh + ch * n[1], wh + ch * n[2], Hh + ch * unh};
  const double R2[5] = {1.0, uh, vh, wh, 0.5 * q2};

  double dut = dU[1] / rhoh - uh * dU[0] / rhoh;
  fence(dut);
  double dvt_ = dU[2] / rhoh - vh * dU[0] / rhoh;
  fence(dvt_);
  double dwt = dU[3] / rhoh - wh * dU[0] / rhoh;
  fence(dwt);
  const double dunf = dut * n[0] + dvt_ * n[1] + dwt * n[2];
  const double tx = dut - dunf * n[0], ty = dvt_ - dunf * n[1], tz = dwt - dunf * n[2];
  double dvt[5] = {0.0, rhoh * tx, rhoh * ty, rhoh * tz, rhoh * (uh * tx + vh * ty + wh * tz)};
  fence(dvt[1], dvt[2], dvt[3], dvt[4]);

  double FL[5], FR[5], absA[5];
  for (int v = 0; v < 5; ++v) absA[v] = al1 * a1 * R1[v] + al5 * a5 * R5[v] + al2 * (a23 * R2[v] + dvt[v]);
  fence(absA[0], absA[1], absA[2], absA[3], absA[4]);
  double VL[5] = {UL[0], UL[1], UL[2], UL[3], UL[4]}, VR[5] = {UR[0], UR[1], UR[2], UR[3], UR[4]};
  fence(VL[0], VL[1], VL[2], VL[3], VL[4]);
  physical_flux(VL, n, g, FL);
  fence(FL[0], FL[1], FL[2], FL[3], FL[4], VR[0], VR[1], VR[2], VR[3], VR[4]);
  physical_flux(VR, n, g, FR);
  for (int v = 0; v < 5; ++v) F[v] = 0.5 * (FL[v] + FR[v]) - 0.5 * absA[v];
}

// One face of rhs/invscd.py:53-97 (the MUSCL-2 slopes of the two cells either
// side, the averaged face metric and the area-weighted Roe flux).  pv0..pv3
// are the primitives of cells a-1, a, a+1, a+2; k0/k1 are kxyz[d, :] at
// cells a and a+1.  Returns F * |n| for the face between a and a+1.
FD void face_flux(const double pv0[5], const double pv1[5], const double pv2[5], const double pv3[5],
                  const double k0[3], const double k1[3], double g, int lim, double Fa[5]) {
  double pL[5], pR[5];
  for (int v = 0; v < 5; ++v) {
    const double sL = limit(lim, pv1[v] - pv0[v], pv2[v] - pv1[v]);
    const double sR = limit(lim, pv2[v] - pv1[v], pv3[v] - pv2[v]);
    pL[v] = pv1[v] + 0.5 * sL;
    pR[v] = pv2[v] - 0.5 * sR;
  }
  double UL[5], UR[5];
  prim_to_cons(pL, g, UL);
  prim_to_cons(pR, g, UR);
  double nf[3] = {0.5 * (k0[0] + k1[0]), 0.5 * (k0[1] + k1[1]), 0.5 * (k0[2] + k1[2])};
  const double nm = sqrt(nf[0] * nf[0] + nf[1] * nf[1] + nf[2] * nf[2]) + 1e-300;
  const double nu[3] = {nf[0] / nm, nf[1] / nm, nf[2] / nm};
  double F[5];
  roe_flux(UL, UR, nu, g, 0.1, F);
  for (int v = 0; v < 5; ++v) Fa[v] = F[v] * nm;
}

// ---------------------------------------------------------------------------
// Stage-kernel forms: the mathematics above, arranged for throughput.
//
// The stage kernels are bound by FP64 issue, so what counts here is the
// number of instructions.  Every product that feeds a sum is an explicit fma
// and the compiler's own contraction is off (EXACT_FP), so a function gives
// the same bits in whichever kernel it is inlined, and the fused and marching
// kernels, which share these functions and the order of every sum, agree bit
// for bit.
// ---------------------------------------------------------------------------

#define DF __device__ __forceinline__
#define EXACT_FP _Pragma("clang fp contract(off)")

// 1/x from the hardware reciprocal seed (relative error e below 2^-24) and
// one cubic correction r (1 + e + e^2): rounding is all that is left (2^-72
// otherwise), in three fma where two Newton steps take four.  For finite
// non-zero x.  (On the host, which checks the arithmetic built on them, this
// and the functions below are the quotient and the root themselves.)
FD double rcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  EXACT_FP
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
#else
  return 1.0 / x;
#endif
}

// sqrt(x) from the hardware reciprocal square-root seed: one cubic correction
// s (1 + e/2 + 3 e^2 / 8), e = 1 - s y measured on the rounded s = x y, then
// the residual x - g^2 of the result, which leaves little but the last rounding
// (without it 0.75 ulp and 0.32 rms instead of 0.50 and 0.29).  IEEE special
// cases: +-0 and +inf are returned as they are (the seed gives inf and 0
// there), x < 0 and NaN give NaN (the seed is NaN).
FD double fsqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  EXACT_FP
  const double y = __builtin_amdgcn_rsq(x);
  const double s = x * y;
  const double e = fma(-s, y, 1.0);
  const double g0 = fma(s * e, fma(e, 0.375, 0.5), s);
  const double g = fma(fma(-g0, g0, x), 0.5 * y, g0);
  // one class test: -0, +0, +inf
  return __builtin_amdgcn_class(x, (1 << 5) | (1 << 6) | (1 << 9)) ? x : g;
#else
  return sqrt(x);
#endif
}

// 1/sqrt(x) for x > 0, the same correction on the seed itself; within 2 ulp
// (checked on the GPU).
FD double rsq_acc(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  EXACT_FP
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
#else
  return 1.0 / sqrt(x);
#endif
}

// One Newton step on the hardware seeds (relative error 2^-24 on gfx950, so
// about 2^-47 after the step: at most ~20 ulp, measured on the GPU), for the
// face flux, whose every quotient and root enters the flux at O(1) weight.
FD double rcp1(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  EXACT_FP
  const double r = __builtin_amdgcn_rcp(x);
  return fma(r, fma(-x, r, 1.0), r);
#else
  return 1.0 / x;
#endif
}
FD double rsq1(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  EXACT_FP
  const double y = __builtin_amdgcn_rsq(x);
  return fma(y * fma(-(x * y), y, 1.0), 0.5, y);
#else
  return 1.0 / sqrt(x);
#endif
}

// van Leer with the division as a reciprocal (stage-kernel form); FULL corrects
// the quotient by its residual: rounded once, like a division
template <bool FULL = false>
FD double vanleer_fast(double a, double b) {
  EXACT_FP
  const double ab = a + b;
  const double safe = fabs(ab) > 1e-30 ? ab : 1.0;
  const double n = 2.0 * a * b, ri = rcp(safe);
  double r = n * ri;
  if constexpr (FULL) r = fma(fma(-safe, r, n), ri, r);
  return (a * b > 0.0) ? r : 0.0;
}

DF void cons_to_prim_fast(const double q[5], double g, double pv[5]) {
  const double rho = q[0];
  const double r = rcp(rho);
  const double u = q[1] * r, v = q[2] * r, w = q[3] * r;
  const double ke = 0.5 * (u * u + v * v + w * w);
  pv[0] = rho; pv[1] = u; pv[2] = v; pv[3] = w;
  pv[4] = (g - 1.0) * (q[4] - rho * ke);
}

// The gas constants the stage kernels use, computed once on the host and held
// in scalar registers (no conversion of them is left in a kernel).
struct StageGas {
  double gm1;      // gamma - 1
  double gm1h;     // (gamma - 1) / 2
  double cg2;      // 2 gamma / (gamma - 1)
  double R, rR;    // R and 1 / R
  double Ts;
  double cmu;      // (T0 + Ts) / T0^1.5 (times the block's mu0: Sutherland's factor of T^1.5 / (T + Ts))
  double ckap;     // gamma R / ((gamma - 1) Pr): kappa / mu
};

// x is the same in every lane of a wave: held in scalar registers
DF double uniform(double x) {
  typedef int pair2 __attribute__((__vector_size__(8)));
  pair2 u = __builtin_bit_cast(pair2, x);
  u[0] = __builtin_amdgcn_readfirstlane(u[0]);
  u[1] = __builtin_amdgcn_readfirstlane(u[1]);
  return __builtin_bit_cast(double, u);
}

// Primitives (rho, u, v, w, p) and temperature of one cell
// (physics/eos.py:12-17, rhs/viscous.py:36) from one reciprocal: 1/rho gives
// the velocities and, with 1/R, the temperature; its floor
// p / max(rho R, 1e-300) is p * 1e300 wherever rho R does not exceed 1e-300.
DF void prim_and_temp(const double q[5], const StageGas& gas, double pv[6]) {
  EXACT_FP
  const double r = rcp(q[0]);
  pv[0] = q[0];
  pv[1] = q[1] * r;
  pv[2] = q[2] * r;
  pv[3] = q[3] * r;
  const double m2 = fma(q[3], pv[3], fma(q[2], pv[2], q[1] * pv[1]));
  pv[4] = gas.gm1 * fma(-0.5, m2, q[4]);
  pv[5] = pv[4] * (q[0] * gas.R > 1e-300 ? r * gas.rR : 1e300);
}

// Twice the area-weighted Roe flux (flux/roe.py:21-85 times |n| + 1e-300,
// rhs/invscd.py:53-97) between the reconstructed primitives pl and pr
// (rho, u, v, w, p) of a face with area vector S (not normalised).  Twice,
// because the factor 1/2 of the flux is cheaper in the cell's 1/vol.
//
// The reference builds the jumps of the conservative variables and recovers
// from them, through the Roe average, quantities that the primitives give
// directly.  With a hat for the Roe average these are identities for any
// rho_L, rho_R > 0 (the floored densities included):
//   (g-1) (dE - u^.dm + q^2/2 drho) = dp,   dm.n - u^n drho = rho^ du_n,
//   (dm - u^ drho) / rho^ = du
// so neither the conservative states nor their jumps are formed (and the
// cancellation in the sums on the left does not arise).  The average takes both
// of its weights, a = sqrt(rho_R) / (sqrt(rho_L) + sqrt(rho_R)) and b = 1 - a
// from the same quotient: as H_L + a (H_R - H_L) it would cancel where the left
// state is the lighter one (H is about p / rho, and a near 1), and so would a
// flux gathered about one side.  Gathered by side instead, the momentum flux
//   m_L u_L + m_R u_R - u^ sa - w du + S P
//     = (m_L - b sa + w) u_L + (m_R - a sa - w) u_R + S P
// (m mass fluxes, sa the summed wave strengths, w the shear weight, P all
// terms along the normal) takes three fma per component.  The energy flux is
// that of the two sides, (E + p) u_n, which no root or reciprocal enters, less
// the waves; the contact wave w2 keeps its own q^2 / 2 (with the acoustic
// waves' H^ and w2 (H^ - q^2 / 2) taken off again it would cancel at large
// density jumps).  Working with S instead of the unit normal leaves one
// 1/|S| and no final product with |S|.  Harten's fix |l| < eps: (l^2/eps + eps)
// / 2 is |l| + (eps - |l|)^2 / (2 eps), zero extra where |l| >= eps.  About 140
// instructions and six seeds, 205 and seven in the form with conservative
// jumps.  Error against 113-bit arithmetic over the largest component, random
// faces with p ~ 1, |u| < 0.5, exact seeds, rms: 1.5e-16 at equal densities and
// 3e-16 at a ratio of 1e6 either way (conservative jumps 2.7e-16 and 3.2e-15;
// gathered about the left state 1.9e-16, and 4.4e-11 with that one lighter);
// with one-step seeds 4e-15 and 1.5e-14 (7e-15 and 1.5e-14), and 1.0e-16 between
// states a thousandth apart (6.6e-15; with the energy flux gathered by side, as
// H times a mass flux, 4.5e-15 and with exact seeds 1.3e-16).  The floors
// are min/max, which drop a NaN: a NaN primitive makes the pressure NaN, and
// dp carries it into every component.
// FULL: every root and reciprocal rounded once (ten seeds instead of six), which
// makes the flux as exact as the reference's formulas in IEEE arithmetic or more
// (rms 1.4e-16 to their 2.5e-16 on those faces, 7.3e-16 to 8.8e-16 at twice the
// speed of sound; with reciprocal roots and their squares 9.5e-16 there).
//
// Says whether no floor acted: where one does, the conservative states that the
// reference forms and these identities part company.
template <bool FULL = false>
FD bool roe_flux2(const double pl[5], const double pr[5], const double S[3], const StageGas& gas, double F[5]) {
  EXACT_FP
  auto recip = [](double x) { return FULL ? rcp(x) : rcp1(x); };
  const double rhoL = fmax(pl[0], 1e-300), rhoR = fmax(pr[0], 1e-300);
  double sqL, sqR, irL, irR;                                      // sqrt(rho), 1 / rho
  if constexpr (FULL) {
    sqL = fsqrt(rhoL), sqR = fsqrt(rhoR);
    irL = rcp(rhoL), irR = rcp(rhoR);
  } else {
    const double isL = rsq1(rhoL), isR = rsq1(rhoR);
    sqL = rhoL * isL, sqR = rhoR * isR;
    irL = isL * isL, irR = isR * isR;
  }
  const double rs = recip(sqL + sqR);
  const double a = sqR * rs, b = sqL * rs;
  const double uL = pl[1], vL = pl[2], wL = pl[3], uR = pr[1], vR = pr[2], wR = pr[3];
  // twice E + p, 2 g/(g-1) p + rho |u|^2, and twice the total enthalpies
  const double kL = fma(wL, wL, fma(vL, vL, uL * uL)), kR = fma(wR, wR, fma(vR, vR, uR * uR));
  const double hL = fma(rhoL, kL, gas.cg2 * pl[4]), hR = fma(rhoR, kR, gas.cg2 * pr[4]);
  const double HL = hL * irL, HR = hR * irR;
  const double uh = fma(a, uR, b * uL), vh = fma(a, vR, b * vL), wh = fma(a, wR, b * wL), Hh = fma(a, HR, b * HL);
  const double q2 = fma(wh, wh, fma(vh, vh, uh * uh));
  const double c2raw = gas.gm1h * (Hh - q2), c2 = fmax(c2raw, 1e-30);
  // |S| and 1/|S|; a zero face keeps a harmless 1e-140
  const double nnraw = fma(S[2], S[2], fma(S[1], S[1], S[0] * S[0])), nn = fmax(nnraw, 1e-280);
  double c, rc2, A, rA;                                           // rc2 = 1 / c^2
  if constexpr (FULL) {
    c = fsqrt(c2), rc2 = rcp(c2);
    A = fsqrt(nn), rA = rcp(A);
  } else {
    const double isc = rsq1(c2);
    rc2 = isc * isc, c = c2 * isc;
    rA = rsq1(nn), A = nn * rA;
  }
  const double C = c * A;
  const double unL = fma(wL, S[2], fma(vL, S[1], uL * S[0])), unR = fma(wR, S[2], fma(vR, S[1], uR * S[0]));
  const double un = fma(a, unR, b * unL);
  const double base = fabs(un) + C;                              // eps = 0.1 base
  const double h = recip(0.2 * base);                             // 1 / (2 eps)
  const double l1 = un - C, l5 = un + C;
  const double e1 = fmax(fma(0.1, base, -fabs(l1)), 0.0), e5 = fmax(fma(0.1, base, -fabs(l5)), 0.0);
  const double al1 = fma(e1 * h, e1, fabs(l1)), al5 = fma(e5 * h, e5, fabs(l5));
  const double dun = (unR - unL) * rA;
  const double dp = pr[4] - pl[4];
  const double rcd = rhoL * rhoR * c * dun;                      // rho^ c (rho^ du_n)
  const double hc = 0.5 * rc2;
  const double w1 = al1 * ((dp - rcd) * hc), w5 = al5 * ((dp + rcd) * hc);
  const double aun = fabs(un);
  const double w2 = aun * fma(-dp, rc2, rhoR - rhoL), w = aun * (sqL * sqR);
  const double sw = w1 + w5, sa = sw + w2;
  const double Q = fma(w, dun, (w1 - w5) * c) * rA;
  const double P = (pl[4] + pr[4]) + Q;
  const double mL = rhoL * unL, mR = rhoR * unR;
  const double iL = fma(-b, sa, mL) + w, iR = fma(-a, sa, mR) - w;
  F[0] = (mL + mR) - sa;
  F[1] = fma(S[0], P, fma(iR, uR, iL * uL));
  F[2] = fma(S[1], P, fma(iR, vR, iL * vL));
  F[3] = fma(S[2], P, fma(iR, wR, iL * wL));
  const double ud = fma(wh, wR - wL, fma(vh, vR - vL, uh * (uR - uL)));
  F[4] = fma(0.5, fma(-w2, q2, fma(-sw, Hh, fma(hR, unR, hL * unL))), fma(un, Q, -(w * ud)));
  return pl[0] > 1e-300 && pr[0] > 1e-300 && c2raw > 1e-30 && nnraw > 1e-280;
}

// MUSCL-2 face states of one cell along one axis (physics/reconstruct/
// muscl2.py:18-37) from the primitives of the cell (pv) and its neighbours
// (pvm below, pvp above): with the limited slope s = lim(pv - pvm, pvp - pv),
// the left state of the cell's high face is pv + s/2 and the right state of
// its low face pv - s/2 -- the slope face_states_fast evaluates once for each of
// the two faces, here once.  The minmod form carries the NaN of the cell two
// away from each face in, as face_states_fast does.
template <int LIM>
FD void muscl_cell(const double pvm[5], const double pv[5], const double pvp[5], double pLhi[5], double pRlo[5]) {
  EXACT_FP
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double am = pv[v] - pvm[v], ap = pvp[v] - pv[v];
    double s;
    if constexpr (LIM == LIM_VANLEER) s = vanleer_fast(am, ap);
    else s = minmod_fast(am, ap);
    pLhi[v] = fma(0.5, s, pv[v]);
    pRlo[v] = fma(-0.5, s, pv[v]);
  }
  if constexpr (LIM == LIM_MINMOD) {
    pLhi[4] = fma(0.0, pvm[4], pLhi[4]);
    pRlo[4] = fma(0.0, pvp[4], pRlo[4]);
  }
}

// The reconstructed states of one face from the primitives of cells a-1, a,
// a+1, a+2 (rhs/invscd.py:53-97).
template <int LIM, bool FULL = false>
FD void face_states_fast(const double pv0[5], const double pv1[5], const double pv2[5], const double pv3[5],
                         double pL[5], double pR[5]) {
  EXACT_FP
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double a = pv1[v] - pv0[v], b = pv2[v] - pv1[v], c = pv3[v] - pv2[v];
    double sL, sR;
    if constexpr (LIM == LIM_VANLEER) {
      sL = vanleer_fast<FULL>(a, b);
      sR = vanleer_fast<FULL>(b, c);
    } else {
      double lo, hi;
      minmod_range(b, lo, hi);
      sL = minmod_in(a, lo, hi);
      sR = minmod_in(c, lo, hi);
    }
    pL[v] = fma(0.5, sL, pv1[v]);
    pR[v] = fma(-0.5, sR, pv2[v]);
  }
  if constexpr (LIM == LIM_MINMOD) {
    // The reference's minmod is NaN when a slope is, which makes the face
    // flux NaN whenever any primitive of the four cells is NaN (a NaN in
    // pL or pR reaches every flux component through the pressure jump).
    // minmod_in drops NaN, so the NaN of the outer cells is carried in
    // here: a cell with any NaN primitive has a NaN pressure (p is computed
    // from all five conservative variables), and 0 * p is +-0 otherwise.
    // (van Leer selects 0 for a NaN slope in the reference as well.)
    pL[4] = fma(0.0, pv0[4], pL[4]);
    pR[4] = fma(0.0, pv3[4], pR[4]);
  }
}

// Twice the flux of one face (roe_flux2) from the primitives of cells a-1 ..
// a+2 and kxyz[d, :] / 2 at cells a and a+1: the area vector is their sum.
template <int LIM, bool FULL = false>
FD bool face_flux2(const double pv0[5], const double pv1[5], const double pv2[5], const double pv3[5],
                   const double k0h[3], const double k1h[3], const StageGas& gas, double F[5]) {
  EXACT_FP
  double pL[5], pR[5];
  face_states_fast<LIM, FULL>(pv0, pv1, pv2, pv3, pL, pR);
  const double S[3] = {k0h[0] + k1h[0], k0h[1] + k1h[1], k0h[2] + k1h[2]};
  return roe_flux2<FULL>(pL, pR, S, gas, F);
}

// Viscous flux tensor of one cell (rhs/viscous.py:30-108): velocity and
// temperature (u, v, w, T) at the cell, the differences d[l][s] = s(+e_l) -
// s(-e_l) of (u, v, w, T), kh = kxyz / 2 at the cell (the 1/2 of the central
// differences, exact on the metrics), cmu = the block's Sutherland factor.
DF void viscous_flux_fast(const double uvwT[4], const double d[3][4], const double kh[9], double cmu,
                          const StageGas& gas, double G[9]) {
  EXACT_FP
  const double T = uvwT[3];
  const double mu = cmu * (T * fsqrt(T)) * rcp(T + gas.Ts);
  const double mu2 = mu + mu, kappa = gas.ckap * mu;
  double gr[4][3];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int m = 0; m < 3; ++m) gr[s][m] = fma(d[2][s], kh[6 + m], fma(d[1][s], kh[3 + m], d[0][s] * kh[m]));
  const double m3 = mu2 * ((gr[0][0] + gr[1][1] + gr[2][2]) * (1.0 / 3.0));
  const double t00 = fma(mu2, gr[0][0], -m3), t11 = fma(mu2, gr[1][1], -m3), t22 = fma(mu2, gr[2][2], -m3);
  const double t01 = mu * (gr[0][1] + gr[1][0]), t02 = mu * (gr[0][2] + gr[2][0]), t12 = mu * (gr[1][2] + gr[2][1]);
  const double u = uvwT[0], v = uvwT[1], w = uvwT[2];
  G[0] = t00; G[1] = t01; G[2] = t02; G[3] = t11; G[4] = t12; G[5] = t22;
  G[6] = fma(w, t02, fma(v, t01, fma(u, t00, kappa * gr[3][0])));
  G[7] = fma(w, t12, fma(v, t11, fma(u, t01, kappa * gr[3][1])));
  G[8] = fma(w, t22, fma(v, t12, fma(u, t02, kappa * gr[3][2])));
}

// The viscous divergence (rhs/viscous.py:86-108), sum over l, j of kxyz[l, j]
// (G_j(+e_l) - G_j(-e_l)) / 2 for each row, as one running sum per row in a
// fixed order: first the lower i-neighbour's share (visc_div_im: known as
// soon as the cell's metrics are, one plane before the rest), then the j and
// k differences dj, dk, then the upper i-neighbour's.  kh = kxyz / 2.
DF void visc_div_im(const double Gm[9], const double kh[9], double vis[4]);
DF void visc_div_jk(const double dj[9], const double dk[9], const double kh[9], double vis[4]);
DF void visc_div_ip(const double Gp[9], const double kh[9], double vis[4]);

// The update of one cell: vis the viscous divergence, A twice the summed face
// differences (j, then k, then i), rvh = 1 / (2 (vol + 1e-300)); Shu-Osher
// (solver/step.py:45-53) as a q0 + b (qs + dt rhs).
struct StageCoef {
  double a, b, dt;
};
DF StageCoef stage_coef(int stage, double dt) {
  const double a = stage == 1 ? 0.0 : (stage == 2 ? 0.75 : 1.0 / 3.0);
  const double b = stage == 1 ? 1.0 : (stage == 2 ? 0.25 : 2.0 / 3.0);
  return StageCoef{uniform(a), uniform(b), uniform(dt)};
}
DF double stage_update(const StageCoef& sc, double q0, double qs, double A, double rvh, double vis) {
  EXACT_FP
  return fma(sc.b, fma(sc.dt, fma(-A, rvh, vis), qs), sc.a * q0);
}

struct Gas {
  double gamma, R, mu0, T0, Ts, Pr_lam;
};

// rhs/viscous.py:30-108 at one cell: given the primitives of the cell, its
// central differences d[l][s] = 0.5*(s(+e_l) - s(-e_l)) of s in (u,v,w,T) and
// kxyz at the cell, produce the viscous flux tensor G = (tau00, tau01, tau02,
// tau11, tau12, tau22, E0, E1, E2) with E_j = u_i tau_ij - heat_j.
FD void viscous_flux(const double pv[5], double T, const double d[3][4], const double k[9],
                     const Gas& gas, double G[9]) {
  const double mu = sutherland(T, gas.mu0, gas.T0, gas.Ts);
  const double cp = gas.gamma * gas.R / (gas.gamma - 1.0);
  const double kappa = cp * mu / gas.Pr_lam;
  double gr[4][3];  // gr[s][m] = d s / d x_m = sum_l d[l][s] * k[l][m]
  for (int s = 0; s < 4; ++s)
    for (int m = 0; m < 3; ++m)
      gr[s][m] = d[0][s] * k[0 * 3 + m] + d[1][s] * k[1 * 3 + m] + d[2][s] * k[2 * 3 + m];
  const double divu = gr[0][0] + gr[1][1] + gr[2][2];
  const double t00 = 2 * mu * (gr[0][0] - divu / 3.0);
  const double t01 = mu * (gr[0][1] + gr[1][0]);
  const double t02 = mu * (gr[0][2] + gr[2][0]);
  const double t11 = 2 * mu * (gr[1][1] - divu / 3.0);
  const double t12 = mu * (gr[1][2] + gr[2][1]);
  const double t22 = 2 * mu * (gr[2][2] - divu / 3.0);
  const double u = pv[1], v = pv[2], w = pv[3];
  G[0] = t00; G[1] = t01; G[2] = t02; G[3] = t11; G[4] = t12; G[5] = t22;
  G[6] = u * t00 + v * t01 + w * t02 - (-kappa * gr[3][0]);
  G[7] = u * t01 + v * t11 + w * t12 - (-kappa * gr[3][1]);
  G[8] = u * t02 + v * t12 + w * t22 - (-kappa * gr[3][2]);
}

DF double temperature_fast(const double pv[5], double R) { return pv[4] * rcp(max_floor(pv[0] * R, 1e-300)); }

// T = p / max(rho R, 1e-300)  (rhs/viscous.py:36)
FD double temperature(const double pv[5], double R) { return pv[4] / max_floor(pv[0] * R, 1e-300); }

// Tensor component index of G for (row r in 0..3, column j): rows 0..2 are
// tau_rj, row 3 is E_j.
FD int gidx(int r, int j) {
  if (r == 3) return 6 + j;
  const int a = r < j ? r : j, b = r < j ? j : r;
  return a == 0 ? b : (a == 1 ? 2 + b : 5);
}

DF void visc_div_im(const double Gm[9], const double kh[9], double vis[4]) {
  EXACT_FP
#pragma unroll
  for (int r = 0; r < 4; ++r)
    vis[r] = fma(-Gm[gidx(r, 2)], kh[2], fma(-Gm[gidx(r, 1)], kh[1], -Gm[gidx(r, 0)] * kh[0]));
}
DF void visc_div_jk(const double dj[9], const double dk[9], const double kh[9], double vis[4]) {
  EXACT_FP
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const int c = gidx(r, m);
      vis[r] = fma(dk[c], kh[6 + m], fma(dj[c], kh[3 + m], vis[r]));
    }
}
DF void visc_div_ip(const double Gp[9], const double kh[9], double vis[4]) {
  EXACT_FP
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int m = 0; m < 3; ++m) vis[r] = fma(Gp[gidx(r, m)], kh[m], vis[r]);
}

}  // namespace famrdp

// Hand-written reverse-mode derivatives (vector-Jacobian products) of the
// pointwise numerics in famrdp_math.h, for the adjoint of the TVD-RK3 step.
//
// Branches are taken the way jax.grad takes them for the reference code
// (famrdp_jax/...): jnp.where sends the cotangent to the selected branch,
// jnp.maximum/minimum split it 1/2-1/2 on exact ties, jnp.abs has derivative
// select(x >= 0, 1, -1), jnp.sign has derivative 0.  The metric terms (face
// normals, kxyz, vol) are constants of the differentiation.
//
// Functions are host+device so the reverse sweeps can be checked on the CPU;
// on the GPU the reciprocals and square roots use the stage-kernel forms.
#pragma once

#include "famrdp_math.h"

namespace famrdp {

FD double rcp_hd(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return rcp(x);
#else
  return 1.0 / x;
#endif
}

FD double sqrt_hd(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return fsqrt(x);
#else
  return sqrt(x);
#endif
}

// d|x|/dx as JAX takes it
FD double dabs(double x) { return x >= 0.0 ? 1.0 : -1.0; }
// d max(x, c)/dx for a constant floor c (ties split 1/2)
FD double dmax_floor(double x, double c) { return x > c ? 1.0 : (x == c ? 0.5 : 0.0); }

// cons_to_prim (physics/eos.py:12-17) reverse: lp = cotangent of
// (rho, u, v, w, p), q the conservative state; accumulates into lq.
FD void cons_to_prim_vjp(const double q[5], double g, const double lp[5], double lq[5]) {
  const double rho = q[0];
  const double r = rcp_hd(rho);
  const double u = q[1] * r, v = q[2] * r, w = q[3] * r;
  const double ke = 0.5 * (u * u + v * v + w * w);
  const double gm1 = g - 1.0;
  // p = gm1 (q4 - rho ke): dp/dq4 = gm1, dp/drho = -gm1 ke, dp/du = -gm1 rho u
  const double lu = lp[1] - gm1 * rho * u * lp[4];
  const double lv = lp[2] - gm1 * rho * v * lp[4];
  const double lw = lp[3] - gm1 * rho * w * lp[4];
  lq[4] += gm1 * lp[4];
  lq[1] += lu * r;
  lq[2] += lv * r;
  lq[3] += lw * r;
  lq[0] += lp[0] - gm1 * ke * lp[4] - (u * lu + v * lv + w * lw) * r;
}

// Limiter reverse: s = lim(A, B) (physics/reconstruct/muscl2.py:5-12).
template <int LIM>
FD void limiter_vjp_t(double A, double B, double ls, double& lA, double& lB) {
  if constexpr (LIM == LIM_VANLEER) {
    if (A * B > 0.0) {
      const double ab = A + B;
      const bool use = fabs(ab) > 1e-30;
      const double den = use ? ab : 1.0;
      const double rd = rcp_hd(den);
      const double s = 2.0 * A * B * rd;
      lA = ls * (2.0 * B * rd - (use ? s * rd : 0.0));
      lB = ls * (2.0 * A * rd - (use ? s * rd : 0.0));
    } else {
      lA = 0.0; lB = 0.0;
    }
  } else {
    // minmod: s = S min(|A|, |B|), S = sign(A) max(sign(A) sign(B), 0), dS = 0.
    // S is nonzero only when A and B have one strict sign, and then
    // S |.|'(A) = S |.|'(B) = 1: the cotangent goes to the smaller magnitude
    // (split 1/2 on a tie).
    const bool same = (A > 0.0 && B > 0.0) || (A < 0.0 && B < 0.0);
    const double xa = fabs(A), xb = fabs(B);
    const double wa = xa < xb ? 1.0 : (xa == xb ? 0.5 : 0.0);
    const double wb = xb < xa ? 1.0 : (xa == xb ? 0.5 : 0.0);
    lA = same ? ls * wa : 0.0;
    lB = same ? ls * wb : 0.0;
  }
}

FD void limiter_vjp(int lim, double A, double B, double ls, double& lA, double& lB) {
  if (lim == LIM_VANLEER) limiter_vjp_t<LIM_VANLEER>(A, B, ls, lA, lB);
  else limiter_vjp_t<LIM_MINMOD>(A, B, ls, lA, lB);
}

// Reverse of roe_flux2 (famrdp_math.h: twice the area-weighted Roe flux of a
// face with area vector S, from the jumps of the primitives): f = cotangent
// of its five components; the cotangents of the left and right primitives are
// written to lpl, lpr.  The forward values are computed again, with the full
// reciprocals and roots, and swept backwards; the same identities of the Roe
// average that shorten the forward flux leave about 280 instructions where
// the sweep through conservative jumps took 430, and far fewer values alive.
// Roots and reciprocals are rounded once each: with 1/sqrt alone and its square
// for 1/rho and 1/c^2 the error at ordinary densities is a third larger (rms
// 3.6e-16 of the largest cotangent and 2.7e-16 with these, 2.9e-16 through
// conservative jumps; gradients 2 % slower for it).
// Both weights a and b = 1 - a as there; b_a is the cotangent of a with b
// following it.  cg2 = 2 g / (g - 1), gm1h = (g - 1) / 2.
FD void roe_flux2_vjp(const double pl[5], const double pr[5], const double S[3], double cg2, double gm1h,
                      const double f[5], double lpl[5], double lpr[5]) {
  const double rhoL = max_floor(pl[0], 1e-300), rhoR = max_floor(pr[0], 1e-300);
  const double sqL = sqrt_hd(rhoL), sqR = sqrt_hd(rhoR);
  const double rs = rcp_hd(sqL + sqR);
  const double a = sqR * rs, b = sqL * rs;
  const double irL = rcp_hd(rhoL), irR = rcp_hd(rhoR);
  const double isL = sqL * irL, isR = sqR * irR;
  const double HL = cg2 * (pl[4] * irL) + (pl[1] * pl[1] + pl[2] * pl[2] + pl[3] * pl[3]);
  const double HR = cg2 * (pr[4] * irR) + (pr[1] * pr[1] + pr[2] * pr[2] + pr[3] * pr[3]);
  double du[3], uh[3];
  for (int m = 0; m < 3; ++m) {
    du[m] = pr[1 + m] - pl[1 + m];
    uh[m] = a * pr[1 + m] + b * pl[1 + m];
  }
  const double Hh = a * HR + b * HL;
  const double q2 = uh[0] * uh[0] + uh[1] * uh[1] + uh[2] * uh[2];
  const double c2raw = gm1h * (Hh - q2);
  const double c2 = max_floor(c2raw, 1e-30);
  const double rc2 = rcp_hd(c2), c = sqrt_hd(c2);
  const double nn0 = S[0] * S[0] + S[1] * S[1] + S[2] * S[2];
  const double nn = nn0 > 1e-280 ? nn0 : 1e-280;
  const double A = sqrt_hd(nn), rA = rcp_hd(A), C = c * A;
  const double unL = pl[1] * S[0] + pl[2] * S[1] + pl[3] * S[2], unR = pr[1] * S[0] + pr[2] * S[1] + pr[3] * S[2];
  const double dS = unR - unL, un = a * unR + b * unL;
  const double aun = fabs(un), sun = dabs(un);
  const double base = aun + C, h = rcp_hd(0.2 * base);
  const double l1 = un - C, l5 = un + C;
  const double x1 = 0.1 * base - fabs(l1), x5 = 0.1 * base - fabs(l5);
  const double e1 = x1 > 0.0 ? x1 : 0.0, e5 = x5 > 0.0 ? x5 : 0.0;
  const double eh1 = e1 * h, eh5 = e5 * h;
  const double al1 = fabs(l1) + eh1 * e1, al5 = fabs(l5) + eh5 * e5;
  const double dun = dS * rA, dp = pr[4] - pl[4], dr = rhoR - rhoL;
  const double rr = rhoL * rhoR, rcd = rr * c * dun, hc = 0.5 * rc2;
  const double a1 = (dp - rcd) * hc, a5 = (dp + rcd) * hc, a23 = dr - dp * rc2;
  const double w1 = al1 * a1, w5 = al5 * a5, w2 = aun * a23, sLR = sqL * sqR, w = aun * sLR;
  const double sw = w1 + w5, sa = sw + w2;
  const double Q = (w * dun + (w1 - w5) * c) * rA;
  const double eL = rhoL * unL - b * sw, eR = rhoR * unR - a * sw;
  const double iL = (eL - b * w2) + w, iR = (eR - a * w2) - w;
  const double ud = uh[0] * du[0] + uh[1] * du[1] + uh[2] * du[2];

  // ---- backwards: momentum and energy components
  const double h4 = 0.5 * f[4];
  const double fu = f[1] * du[0] + f[2] * du[1] + f[3] * du[2];
  const double b_mL = f[0] + (f[1] * pl[1] + f[2] * pl[2] + f[3] * pl[3]) + h4 * HL;
  const double b_mR = f[0] + (f[1] * pr[1] + f[2] * pr[2] + f[3] * pr[3]) + h4 * HR;
  const double b_P = f[1] * S[0] + f[2] * S[1] + f[3] * S[2];
  const double b_ud = -f[4] * w;
  const double b_HL0 = h4 * eL, b_HR0 = h4 * eR;
  double b_un = f[4] * Q;
  const double q = (f[4] * un + b_P) * rA;
  const double b_w = q * dun - f[4] * ud - fu;
  double b_dun = q * w;
  const double b_sa = -(f[0] + (f[1] * uh[0] + f[2] * uh[1] + f[3] * uh[2]));
  const double dH = HR - HL;
  double b_a = -sa * fu - h4 * (sw * dH);
  // ---- wave strengths
  const double b_sw = b_sa - h4 * Hh;
  const double b_w1 = b_sw + q * c, b_w5 = b_sw - q * c, b_w2 = b_sa - h4 * q2;
  double b_c = q * (w1 - w5);
  const double b_aun = b_w2 * a23 + b_w * sLR, b_a23 = b_w2 * aun, b_sLR = b_w * aun;
  const double b_al1 = b_w1 * a1, b_al5 = b_w5 * a5;
  const double t1 = b_w1 * al1, t5 = b_w5 * al5;
  const double b_rcd = (t5 - t1) * hc;
  const double b_dp = (t1 + t5) * hc - b_a23 * rc2;
  // rc2 enters through hc = rc2 / 2 (a1, a5 = (dp -+ rcd) hc) and a23
  const double b_rc2 = 0.5 * (t1 * (dp - rcd) + t5 * (dp + rcd)) - b_a23 * dp;
  b_c += b_rcd * (rr * dun);
  b_dun += b_rcd * (rr * c);
  const double b_rr = b_rcd * (c * dun);
  // ---- Harten's fix: al = |l| + e^2 h, e = max(base / 10 - |l|, 0), h = 5 / base
  const double g1 = b_al1 * (1.0 - 2.0 * eh1) * dabs(l1), g5 = b_al5 * (1.0 - 2.0 * eh5) * dabs(l5);
  const double b_base = 0.2 * (b_al1 * (eh1 * (1.0 - eh1)) + b_al5 * (eh5 * (1.0 - eh5)));
  b_un += (g1 + g5) + (b_base + b_aun) * sun;
  b_c += (b_base + (g5 - g1)) * A;
  // ---- normal velocities
  b_a += b_un * dS;
  const double b_dS = b_dun * rA;
  const double b_unL = (b * b_un - b_dS) + b_mL * rhoL, b_unR = (a * b_un + b_dS) + b_mR * rhoR;
  // ---- sound speed, Roe average
  const double b_c2 = rc2 * (0.5 * b_c * c - b_rc2 * rc2);
  const double b_hq = gm1h * (b_c2 * dmax_floor(c2raw, 1e-30));
  const double b_HL = b_HL0 + b * b_hq, b_HR = b_HR0 + a * b_hq;
  const double b_q2 = -2.0 * (h4 * w2 + b_hq);
  b_a += b_hq * dH;
  double b_rhoL = b_mL * unL + b_rr * rhoR - b_a23, b_rhoR = b_mR * unR + b_rr * rhoL + b_a23;
  for (int m = 0; m < 3; ++m) {
    const double b_uh = b_ud * du[m] + b_q2 * uh[m], b_du = b_ud * uh[m];
    b_a += b_uh * du[m];
    lpl[1 + m] = iL * f[1 + m] + (b * b_uh - b_du) + b_unL * S[m] + 2.0 * b_HL * pl[1 + m];
    lpr[1 + m] = iR * f[1 + m] + (a * b_uh + b_du) + b_unR * S[m] + 2.0 * b_HR * pr[1 + m];
  }
  const double cL = b_HL * cg2 * irL, cR = b_HR * cg2 * irR;
  lpl[4] = b_P - b_dp + cL;
  lpr[4] = b_P + b_dp + cR;
  const double b_s = b_a * rs;                 // a = sqR / (sqL + sqR)
  const double b_sL = b_sLR * sqR - b_s * a, b_sR = b_sLR * sqL + b_s * b;
  b_rhoL += 0.5 * b_sL * isL - cL * (pl[4] * irL);
  b_rhoR += 0.5 * b_sR * isR - cR * (pr[4] * irR);
  lpl[0] = b_rhoL * dmax_floor(pl[0], 1e-300);
  lpr[0] = b_rhoR * dmax_floor(pr[0], 1e-300);
}

// The same for the flux itself with a unit normal (flux/roe.py:21-85),
// accumulating into lpl, lpr.
FD void roe_flux_prim_vjp(const double pl[5], const double pr[5], const double n[3], double g, const double lF[5],
                          double lpl[5], double lpr[5]) {
  double f[5], bl[5], br[5];
  for (int v = 0; v < 5; ++v) f[v] = 0.5 * lF[v];
  roe_flux2_vjp(pl, pr, n, 2.0 * g / (g - 1.0), 0.5 * (g - 1.0), f, bl, br);
  for (int v = 0; v < 5; ++v) {
    lpl[v] += bl[v];
    lpr[v] += br[v];
  }
}

// Viscous flux tensor (rhs/viscous.py:30-108) reverse.  Inputs as
// viscous_flux; lG = cotangent of G[9]; outputs accumulate the cotangents of
// u, v, w (direct use in the energy flux), T (through mu and kappa) and the
// central differences d[l][s].
FD void viscous_flux_vjp(const double pv[5], double T, const double d[3][4], const double k[9], double gamma,
                         double R, double mu0, double T0, double Ts, double Pr, const double lG[9], double& lu,
                         double& lv, double& lw, double& lT, double ld[3][4]) {
  const double x = T * rcp_hd(T0);
  const double sx = sqrt_hd(x);
  const double rTs = rcp_hd(T + Ts);
  const double mu = mu0 * (x * sx) * (T0 + Ts) * rTs;
  const double cp_pr = gamma * R * rcp_hd(gamma - 1.0) * rcp_hd(Pr);
  const double kappa = cp_pr * mu;
  double gr[4][3];
  for (int s = 0; s < 4; ++s)
    for (int m = 0; m < 3; ++m) gr[s][m] = d[0][s] * k[0 * 3 + m] + d[1][s] * k[1 * 3 + m] + d[2][s] * k[2 * 3 + m];
  const double divu3 = (gr[0][0] + gr[1][1] + gr[2][2]) * (1.0 / 3.0);
  const double t00 = 2 * mu * (gr[0][0] - divu3), t01 = mu * (gr[0][1] + gr[1][0]), t02 = mu * (gr[0][2] + gr[2][0]);
  const double t11 = 2 * mu * (gr[1][1] - divu3), t12 = mu * (gr[1][2] + gr[2][1]), t22 = 2 * mu * (gr[2][2] - divu3);
  const double u = pv[1], v = pv[2], w = pv[3];
  // E_j = u t0j + v t1j + w t2j + kappa dT/dx_j
  const double b00 = lG[0] + u * lG[6];
  const double b01 = lG[1] + v * lG[6] + u * lG[7];
  const double b02 = lG[2] + w * lG[6] + u * lG[8];
  const double b11 = lG[3] + v * lG[7];
  const double b12 = lG[4] + w * lG[7] + v * lG[8];
  const double b22 = lG[5] + w * lG[8];
  lu += t00 * lG[6] + t01 * lG[7] + t02 * lG[8];
  lv += t01 * lG[6] + t11 * lG[7] + t12 * lG[8];
  lw += t02 * lG[6] + t12 * lG[7] + t22 * lG[8];
  const double b_kappa = gr[3][0] * lG[6] + gr[3][1] * lG[7] + gr[3][2] * lG[8];
  double bg[4][3];
  bg[3][0] = kappa * lG[6]; bg[3][1] = kappa * lG[7]; bg[3][2] = kappa * lG[8];
  const double b_mu = 2.0 * (gr[0][0] - divu3) * b00 + (gr[0][1] + gr[1][0]) * b01 + (gr[0][2] + gr[2][0]) * b02 +
                      2.0 * (gr[1][1] - divu3) * b11 + (gr[1][2] + gr[2][1]) * b12 +
                      2.0 * (gr[2][2] - divu3) * b22 + cp_pr * b_kappa;
  const double b_div3 = -2.0 * mu * (b00 + b11 + b22);
  bg[0][0] = 2.0 * mu * b00 + b_div3 * (1.0 / 3.0);
  bg[1][1] = 2.0 * mu * b11 + b_div3 * (1.0 / 3.0);
  bg[2][2] = 2.0 * mu * b22 + b_div3 * (1.0 / 3.0);
  bg[0][1] = mu * b01; bg[1][0] = mu * b01;
  bg[0][2] = mu * b02; bg[2][0] = mu * b02;
  bg[1][2] = mu * b12; bg[2][1] = mu * b12;
  for (int l = 0; l < 3; ++l)
    for (int s = 0; s < 4; ++s)
      ld[l][s] += bg[s][0] * k[l * 3 + 0] + bg[s][1] * k[l * 3 + 1] + bg[s][2] * k[l * 3 + 2];
  // mu = mu0 x^1.5 (T0+Ts)/(T+Ts):  dmu/dT = mu (1.5/T - 1/(T+Ts))
  lT += b_mu * mu * (1.5 * rcp_hd(T) - rTs);
}

// T = p / max(rho R, 1e-300) reverse into (rho, p).
FD void temperature_vjp(const double pv[5], double R, double lT, double& lrho, double& lp) {
  const double den = pv[0] * R;
  const double dn = max_floor(den, 1e-300);
  const double rd = rcp_hd(dn);
  lp += lT * rd;
  lrho -= lT * pv[4] * rd * rd * R * dmax_floor(den, 1e-300);
}

// No-slip isothermal ghost value (physics/bc/wall.py:35-58) reverse: lo =
// cotangent of the ghost cell, accumulated into li (the mirrored inner cell).
FD void isothermal_vjp(const double qi[5], double gamma, double R, double Tw, const double lo[5], double li[5]) {
  const double gm1 = gamma - 1.0;
  const double rho_i = qi[0];
  const double ssum = qi[1] * qi[1] + qi[2] * qi[2] + qi[3] * qi[3];
  const double ke_i = 0.5 * ssum / rho_i;
  const double p = gm1 * (qi[4] - ke_i);
  const double rho_g = p / (R * Tw);
  const double scale = rho_g / rho_i;
  const double m[3] = {-qi[1] * scale, -qi[2] * scale, -qi[3] * scale};
  const double ke_g = 0.5 * (m[0] * m[0] + m[1] * m[1] + m[2] * m[2]) / rho_g;
  double b_rho_g = lo[0], b_p = lo[4] / gm1, b_keg = lo[4];
  double b_m[3] = {lo[1], lo[2], lo[3]};
  for (int k = 0; k < 3; ++k) b_m[k] += b_keg * m[k] / rho_g;
  b_rho_g -= b_keg * ke_g / rho_g;
  double b_scale = 0.0;
  for (int k = 0; k < 3; ++k) { li[1 + k] -= b_m[k] * scale; b_scale -= b_m[k] * qi[1 + k]; }
  b_rho_g += b_scale / rho_i;
  double b_rho_i = -b_scale * scale / rho_i;
  b_p += b_rho_g / (R * Tw);
  li[4] += gm1 * b_p;
  const double b_kei = -gm1 * b_p;
  for (int k = 0; k < 3; ++k) li[1 + k] += b_kei * qi[1 + k] / rho_i;
  b_rho_i -= b_kei * ke_i / rho_i;
  li[0] += b_rho_i;
}

}  // namespace famrdp

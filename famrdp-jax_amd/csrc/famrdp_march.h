// i-marching stage kernel: one launch per RK3 stage (solver/step.py:45-53),
// the same operator as the fused tile kernel (rhs/invscd.py:53-131,
// rhs/viscous.py:30-108), computed with the same expressions in the same
// order, so both give the same bits.
//
// A workgroup owns a column of TJ x TK cells (one thread per (j, k) column)
// over a segment [pA, pB) of planes along i, the slowest axis, and walks it
// one plane per step, with two barriers per step.  Step s, for s = pA-1 .. pB:
//
//   A. The primitives and temperature of plane s go to the LDS plane P: the
//      tile's columns and two halo rings (the second one without corners),
//      at periodic (roll) coordinates; they were converted in the previous
//      step.  Then what plane s-1 takes from LDS, left there by the previous
//      step: the j and k differences of the viscous tensor G(s-1) and of the
//      j and k face fluxes, and the column's own G(s-1), folded at once into
//      the share the lower i-neighbour of plane s has in its divergence (four
//      values carried instead of nine).  Then the i-face between planes s-1
//      and s of the column, from registers (its left state was reconstructed
//      in the previous step; the right state and the next face's left state
//      share one limited slope per variable).
//   -- barrier: P is in place, and every read of G(s-1) and of its faces done
//   B. G of plane s at the column (j/k differences from P, i differences from
//      the column's registers), which completes the divergence of plane s-1;
//      the Shu-Osher update of plane s-1 is written.  G(s) goes over G(s-1) in
//      LDS, with G of the tile's one-cell cross halo; the MUSCL-2 + Roe faces
//      of plane s along j and k go to the face buffer (each thread its
//      column's low j-face, then its low k-face, both with offsets fixed by
//      the column; the last wave the far-end layer); the halo of plane s+1 is
//      converted for the next step.
//   -- barrier: G(s) and the faces of plane s are in place, P is free
//
// Loads are issued a phase or more before their use and spread through the
// arithmetic (march_spread): the next plane's metrics, the state of the plane
// after it and the update operands through the faces of this plane, the halo's
// state at the end of phase B, the metrics of the faces' other cells and of
// the cross halo at the end of phase A.
//
// What bounds it (260^3 padded, stage 2, random smooth state): neither FP64
// issue nor HBM alone.  The same launch with every load an L2 hit takes
// 1.09 ms, its VALU instructions alone 0.66 ms, its bytes past L2 (6 GB, 1.8
// times the compulsory 3.5 GB: halos, the re-read of the plane being updated)
// 1.2 ms at the 4.9 TB/s of a large copy; at two waves per SIMD (256
// registers, 77.7 KB of LDS) the three overlap to 1.40 ms (132^3: 212 us; with
// the Roe flux gathered about its left state and no residual on the square
// root, 1,229 instead of 1,268 instructions per 64 cells, 1.37 and 211).
// With three barriers per plane, conservative jumps in the Roe flux and the
// far-end faces' loads inside their round: 1.51 ms (231 us).
//
// Each cell's primitives, viscous tensor and faces are computed once per
// segment, apart from the tile's halo rings in j and k and the two extra
// planes at each segment start.  Cell coordinates are fixed per thread for
// the whole march (one plane stride apart from step to step).  Tiles that
// reach past the block in j or k (partial tiles, small blocks) stage and
// compute G at the periodic images of those columns, which is what the
// roll of the viscous terms reads; only columns inside the block write.  A
// narrow k remainder goes to transposed TK x TJ strip tiles (march_tiling),
// so that it does not take a row of TJ x TK tiles owning a few columns each.
// Loads and stores go through buffer resources with 32-bit byte offsets, so
// a block's kxyz must stay under 4 GiB (march_fits).
#pragma once

#include "famrdp_march_geom.h"

namespace famrdp {

// The arrays a march reads and writes, as buffer resources: a load or store
// takes the element's 32-bit byte offset in a vector register and the
// variable's offset v N (bytes) in a scalar register, so no address is formed
// per access (global loads from base + v N formed a 64-bit vector address for
// every variable but the first: 1 % of the stage's time).  Every array of a
// block that march_fits accepts spans fewer than 2^32 bytes, which is the
// resource's record count; the last word is the gfx9-family setting for
// untyped (raw) access (32-bit data format, stride 0).
typedef unsigned march_u2 __attribute__((__vector_size__(8)));

DF __amdgpu_buffer_rsrc_t march_rsrc(const double* p, int64_t n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, (int)(unsigned)(n * 8), 0x00020000);
}

// element i (< 2^29) of variable v: byte offset i * 8 + soff, soff = v N * 8
DF double ldx(__amdgpu_buffer_rsrc_t r, unsigned i, unsigned soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, i << 3, (int)soff, 0));
}

DF void stx(__amdgpu_buffer_rsrc_t r, unsigned i, unsigned soff, double x) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(march_u2, x), r, i << 3, (int)soff, 0);
}

DF void march_load5(__amdgpu_buffer_rsrc_t r, unsigned nb, unsigned off, double x[5]) {
#pragma unroll
  for (int v = 0; v < 5; ++v) x[v] = ldx(r, off, v * nb);
}

// kxyz of the largest block a marching launch may address (9 N doubles
// under 4 GiB)
__host__ __device__ __forceinline__ bool march_fits(int64_t N) { return N * 72 < (int64_t(1) << 32); }

// Viscous flux tensor of the cell at P slot `sl` (rhs/viscous.py:30-108):
// j/k neighbours from P, i neighbours (u, v, w, T) from um (plane s-1) and up
// (plane s+1); kch = kxyz / 2 at the cell.
template <int TJ, int TK>
DF void march_visc(const double* sP, int sl, const double um[4], const double up[4], const double kch[9], double cmu,
                   const StageGas& gas, double g9[9]) {
  EXACT_FP
  using M = MarchGeom<TJ, TK>;
  constexpr int NP = M::NP;
  const double uvwT[4] = {sP[NP + sl], sP[2 * NP + sl], sP[3 * NP + sl], sP[5 * NP + sl]};
  double d[3][4];
#pragma unroll
  for (int s = 0; s < 4; ++s) d[0][s] = up[s] - um[s];
#pragma unroll
  for (int l = 1; l < 3; ++l) {
    const int sp = l == 1 ? sl + M::PK : sl + 1;
    const int sm = l == 1 ? sl - M::PK : sl - 1;
    d[l][0] = sP[NP + sp] - sP[NP + sm];
    d[l][1] = sP[2 * NP + sp] - sP[2 * NP + sm];
    d[l][2] = sP[3 * NP + sp] - sP[3 * NP + sm];
    d[l][3] = sP[5 * NP + sp] - sP[5 * NP + sm];
  }
  viscous_flux_fast(uvwT, d, kch, cmu, gas, g9);
}

// One j- or k-face of the plane (rhs/invscd.py:53-97, twice the flux) into
// face buffer slot f: the four cells' primitives from P slots base + s str
// (s = 0..3), kl, kr = kxyz / 2 of the face's axis at the cells either side.
template <int TJ, int TK, int LIM>
DF void march_face(const double* sP, double* sF, int base, int str, const double kl[3], const double kr[3], int f,
                   const StageGas& gas) {
  using M = MarchGeom<TJ, TK>;
  double p4[4][5];
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) {
#pragma unroll
    for (int v = 0; v < 5; ++v) p4[s4][v] = sP[v * M::NP + base + s4 * str];
  }
  double Fa[5];
  face_flux2<LIM>(p4[0], p4[1], p4[2], p4[3], kl, kr, gas, Fa);
#pragma unroll
  for (int v = 0; v < 5; ++v) sF[v * M::NFB + f] = Fa[v];
}

// v, hidden from the optimiser: what is computed from it inside the march
// loop is computed there, not hoisted out and held in registers
__device__ __forceinline__ unsigned march_opaque(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

// x is computed by here: the compiler moves arithmetic that only a later
// phase consumes past barriers and scheduling fences, down to its use, and
// then holds that arithmetic's many operands in registers instead of x
DF void march_pin(double& x) { asm volatile("" : "+v"(x)); }
template <int K>
DF void march_pin(double (&x)[K]) {
#pragma unroll
  for (int i = 0; i < K; ++i) march_pin(x[i]);
}

// Order for the scheduler: N loads, each followed by V arithmetic
// instructions.  Issued back to back the loads of a phase hold every wave of
// the workgroup at the address unit (about 16 cycles a load and CU, all four
// waves in the same phase); spread through a face they cost their issue slot.
template <int N, int V>
DF void march_spread() {
  if constexpr (N > 0) {
    __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);   // a VMEM read
    __builtin_amdgcn_sched_group_barrier(0x2, V, 0);    // V VALU instructions
    march_spread<N - 1, V>();
  }
}

template <int TJ, int TK, int LIM>
__device__ __forceinline__ void march_segment(double* lds, const BlockDesc& b, int j0, int k0, int pA, int pB,
                                              const double* __restrict__ qin, const double* q0, double* qout,
                                              const StageGas& gas, double dt, int stage) {
  EXACT_FP
  using M = MarchGeom<TJ, TK>;
  double* sP = lds;                          // [6][NP]  rho u v w p T of plane s
  double* sG = sP + 6 * M::NP;               // [9][NGP] G of plane s-1 (then s)
  double* sF = sG + 9 * M::NGP;              // [5][NFB] j/k faces of plane s-1 (then s)
  double* sH = sF + 5 * M::NFB;              // [6][NHS] halo of the next plane
  double* sU = sH + 6 * M::NHS;              // [4][NHG] u v w T of plane s-1 at the G cross halo
  const int t = threadIdx.x;
  const int ni = b.ni, nj = b.nj, nk = b.nk;
  const int64_t N = b.N;
  const unsigned si = (unsigned)nj * (unsigned)nk;
  const double cmu = uniform(gas.cmu * b.mu0);
  const StageCoef sc = stage_coef(stage, dt * b.dt_scale);
  const unsigned nb = (unsigned)N * 8u;     // bytes between variables
  const __amdgpu_buffer_rsrc_t rq = march_rsrc(qin, 5 * N), r0 = march_rsrc(q0, stage == 1 ? 0 : 5 * N),   // stage 1 takes no q0: loads give 0
                               ro = march_rsrc(qout, 5 * N), rk = march_rsrc(b.kxyz, 9 * N),
                               rv = march_rsrc(b.vol, N);

  // ---- fixed per thread for the whole march --------------------------------
  const MarchThread th = M::thread(t, j0, k0, nj, nk);
  const int tj = th.tj, tk = th.tk, slot = th.slot, gslot = th.gslot, hs = th.hs;
  int hslot = th.hslot, hgslot = th.hgslot;
  const bool own = th.own, jin = th.jin, kin = th.kin, hg = th.hg;
  const unsigned col = th.col;
  unsigned hcol = th.hcol, hcol2 = th.hcol;
  // The last wave stages no halo; its threads take the far-end faces (face_of
  // round 2: j-faces past the tile's last row, k-faces past its last column)
  // instead.  The same registers hold their fixed places: hslot the P slot of
  // the cell two before the face, hgslot the face buffer slot, hcol and hcol2
  // the offsets in kxyz of the face's axis at the cells either side (hcol2
  // less the three rows that follow), so the metrics of a far face and of a
  // cross-halo cell are the same loads.
  int fstr = 0;
  const int ff = M::face_of(t, 2);
  if (ff >= 0) {
    const MarchFace fc = M::face(ff, j0, k0, nj, nk);
    if (fc.ok) {
      fstr = fc.str;
      hslot = fc.base;
      hgslot = ff;
      const unsigned row = (fc.isj ? 3u : 6u) * (unsigned)N;
      hcol = row + (fc.isj ? (unsigned)fc.a * nk + fc.oc : (unsigned)fc.oc * nk + fc.a);
      hcol2 = hcol + (fc.isj ? (unsigned)nk : 1u) - 3u * (unsigned)N;
    }
  }
  const bool hm = hg || fstr > 0;   // loads metrics for phase B's last part
  // where the low faces' other cells lie (this cell where there is no face:
  // a valid address, and a flux that no update reads)
  const unsigned dfj = th.fj ? (unsigned)nk : 0u, dfk = th.fk ? 1u : 0u;
  auto plane = [&](int s) -> unsigned { return (unsigned)(s < 0 ? s + ni : (s >= ni ? s - ni : s)) * si; };

  // ---- warm-up: planes pA-2, pA-1 converted, pA loading ---------------------
  double pm[6], pc[6];
  {
    double qq[5], x[6];
    march_load5(rq, nb, plane(pA - 2) + col, qq);
    prim_and_temp(qq, gas, pm);
    march_load5(rq, nb, plane(pA - 1) + col, qq);
    prim_and_temp(qq, gas, pc);
    if (hg) {
      march_load5(rq, nb, plane(pA - 2) + hcol, qq);
      prim_and_temp(qq, gas, x);
      sU[hs] = x[1];
      sU[M::NHG + hs] = x[2];
      sU[2 * M::NHG + hs] = x[3];
      sU[3 * M::NHG + hs] = x[5];
    }
    if (hs >= 0) {
      march_load5(rq, nb, plane(pA - 1) + hcol, qq);
      prim_and_temp(qq, gas, x);
#pragma unroll
      for (int v = 0; v < 6; ++v) sH[v * M::NHS + hs] = x[v];
    }
  }
  double qn[5], kk[9];
  march_load5(rq, nb, plane(pA) + col, qn);
#pragma unroll
  for (int m = 0; m < 9; ++m) kk[m] = ldx(rk, plane(pA - 1) + col, m * nb);

  // the update operands of the next step, and the state of its halo
  double vl = 1.0, qs[5] = {0, 0, 0, 0, 0}, qq0[5] = {0, 0, 0, 0, 0}, qnh[5] = {0, 0, 0, 0, 0};
  if (hs >= 0) march_load5(rq, nb, plane(pA) + hcol, qnh);

  double kpvh[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};   // kxyz / 2 of the column at plane s-1
  double pLn[5] = {0, 0, 0, 0, 0};       // left state of the column's next i-face
  double Fm[5] = {0, 0, 0, 0, 0};        // i-face below plane s-1
  double vism[4] = {0, 0, 0, 0};         // G(s-2)'s share of the divergence of plane s-1

  for (int s = pA - 1; s <= pB; ++s) {
    const unsigned op = plane(s), om = plane(s - 1);
    const unsigned c_s = op + march_opaque(col), c_m = om + march_opaque(col);
    const bool faces = s >= pA && s < pB;            // plane s is owned: its j/k faces
    const bool iin = s - 1 >= 2 && s - 1 <= ni - 3;  // plane s-1 takes its i-faces

    // ---- A. P <- plane s -------------------------------------------------------
#pragma unroll
    for (int v = 0; v < 6; ++v) sP[v * M::NP + slot] = pc[v];
    if (hs >= 0) {
#pragma unroll
      for (int v = 0; v < 6; ++v) sP[v * M::NP + hslot] = sH[v * M::NHS + hs];
    }
    __builtin_amdgcn_sched_barrier(0);
    // what plane s-1 takes from LDS
    double vis[4] = {vism[0], vism[1], vism[2], vism[3]};
    double A[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    {
      double dj[9], dk[9];
#pragma unroll
      for (int m = 0; m < 9; ++m) {
        const double* Gc = sG + m * M::NGP;
        dj[m] = Gc[gslot + M::GK] - Gc[gslot - M::GK];
        dk[m] = Gc[gslot + 1] - Gc[gslot - 1];
      }
      visc_div_jk(dj, dk, kpvh, vis);
      const int lo = tj * TK + tk, lok = M::NFJ + tj * (TK + 1) + tk;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double* Fv = sF + v * M::NFB;
        const double fj = Fv[lo + TK] - Fv[lo], fk = Fv[lok + 1] - Fv[lok];
        A[v] = jin ? fj : 0.0;
        A[v] = kin ? A[v] + fk : A[v];
      }
      march_pin(vis);
      march_pin(A);
    }
    double kkh[9];   // kxyz / 2 of plane s
#pragma unroll
    for (int m = 0; m < 9; ++m) kkh[m] = 0.5 * kk[m];
    {
      double gm[9];
#pragma unroll
      for (int m = 0; m < 9; ++m) gm[m] = sG[m * M::NGP + gslot];
      visc_div_im(gm, kkh, vism);
      march_pin(vism);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the i-face between planes s-1 and s
    double pn[6];
    prim_and_temp(qn, gas, pn);
    {
      double pLs[5], pRs[5], Fi[5];
      muscl_cell<LIM>(pm, pc, pn, pLs, pRs);
      const double S[3] = {kpvh[0] + kkh[0], kpvh[1] + kkh[1], kpvh[2] + kkh[2]};
      roe_flux2(pLn, pRs, S, gas, Fi);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        if (iin) A[v] = A[v] + (Fi[v] - Fm[v]);
        Fm[v] = Fi[v];
        pLn[v] = pLs[v];
      }
      march_pin(A);
      march_pin(Fm);
      march_pin(pLn);
    }
    // metrics of the faces' other cells, and of the cross halo or a far face
    double kh[9], klj[3], klk[3];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      klj[m] = ldx(rk, c_s - dfj, (3 + m) * nb);
      klk[m] = ldx(rk, c_s - dfk, (6 + m) * nb);
    }
    if (hm) {
      const unsigned ch = op + march_opaque(hcol), ch2 = op + march_opaque(hcol2);
#pragma unroll
      for (int m = 0; m < 3; ++m) kh[m] = ldx(rk, ch, m * nb);
#pragma unroll
      for (int m = 3; m < 9; ++m) kh[m] = ldx(rk, ch2, m * nb);
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();   // P in place; G(s-1) and the faces of plane s-1 read
    __builtin_amdgcn_sched_barrier(0);

    // ---- B. G(s), the update of plane s-1 ---------------------------------------
    {
      double g9[9];
      const double um[4] = {pm[1], pm[2], pm[3], pm[5]}, up[4] = {pn[1], pn[2], pn[3], pn[5]};
      march_visc<TJ, TK>(sP, slot, um, up, kkh, cmu, gas, g9);
      visc_div_ip(g9, kpvh, vis);
#pragma unroll
      for (int m = 0; m < 9; ++m) sG[m * M::NGP + gslot] = g9[m];
      march_pin(vis);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (s > pA && own) {   // plane s-1 is the segment's (s-1 < pB always)
      const double rvh = 0.5 * rcp(vl + 1e-300);
#pragma unroll
      for (int v = 0; v < 5; ++v)
        stx(ro, c_m, v * nb, stage_update(sc, qq0[v], qs[v], A[v], rvh, v == 0 ? 0.0 : vis[v - 1]));
    }
#pragma unroll
    for (int v = 0; v < 6; ++v) {
      pm[v] = pc[v];
      pc[v] = pn[v];
    }
#pragma unroll
    for (int m = 0; m < 9; ++m) kpvh[m] = kkh[m];
    __builtin_amdgcn_sched_barrier(0);
    // G of the cross halo; the next plane's halo
    if (hs >= 0) {
      double x[6];
      prim_and_temp(qnh, gas, x);     // plane s+1 at the halo cell
#pragma unroll
      for (int v = 0; v < 6; ++v) sH[v * M::NHS + hs] = x[v];
      if (hg) {
        const double um[4] = {sU[hs], sU[M::NHG + hs], sU[2 * M::NHG + hs], sU[3 * M::NHG + hs]};
        const double up[4] = {x[1], x[2], x[3], x[5]};
        double khh[9], g9h[9];
#pragma unroll
        for (int m = 0; m < 9; ++m) khh[m] = 0.5 * kh[m];
        march_visc<TJ, TK>(sP, hslot, um, up, khh, cmu, gas, g9h);
#pragma unroll
        for (int m = 0; m < 9; ++m) sG[m * M::NGP + hgslot] = g9h[m];
        sU[hs] = sP[M::NP + hslot];
        sU[M::NHG + hs] = sP[2 * M::NP + hslot];
        sU[2 * M::NHG + hs] = sP[3 * M::NP + hslot];
        sU[3 * M::NHG + hs] = sP[5 * M::NP + hslot];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next plane's metrics and the state of the plane after it, and the
    // update operands of plane s; loaded on either side of `faces`, so that no
    // older value has to be kept for a step that does not need them
    auto load_next = [&] {
#pragma unroll
      for (int m = 0; m < 9; ++m) kk[m] = ldx(rk, plane(s + 1) + march_opaque(col), m * nb);
      march_load5(rq, nb, plane(s + 2) + march_opaque(col), qn);
    };
    auto load_operands = [&] {
      vl = ldx(rv, op + march_opaque(col), 0);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        qs[v] = ldx(rq, op + march_opaque(col), v * nb);
        qq0[v] = ldx(r0, op + march_opaque(col), v * nb);
      }
    };
    if (!faces) load_next();
    if (faces) {
      double klh[3];
      // round 0: the column's low j-face (cells gj-2 .. gj+1 of column gk),
      // between its instructions load_operands
#pragma unroll
      for (int m = 0; m < 3; ++m) klh[m] = 0.5 * klj[m];
      load_operands();
      march_face<TJ, TK, LIM>(sP, sF, slot - 2 * M::PK, M::PK, klh, kpvh + 3, t, gas);
      march_spread<11, 16>();
      __builtin_amdgcn_sched_barrier(0);   // one face at a time: the rounds are not interleaved
      // round 1: the column's low k-face, between its instructions load_next
#pragma unroll
      for (int m = 0; m < 3; ++m) klh[m] = 0.5 * klk[m];
      load_next();
      march_face<TJ, TK, LIM>(sP, sF, slot - 2, 1, klh, kpvh + 6, M::NFJ + tj * (TK + 1) + tk, gas);
      march_spread<14, 13>();
      __builtin_amdgcn_sched_barrier(0);
      if (fstr > 0) {   // round 2: the far-end layer
        double kl[3], kr[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          kl[m] = 0.5 * kh[m];
          kr[m] = 0.5 * kh[3 + m];
        }
        march_face<TJ, TK, LIM>(sP, sF, hslot, fstr, kl, kr, hgslot, gas);
      }
    }
    if (!faces) load_operands();
    if (hs >= 0) march_load5(rq, nb, plane(s + 2) + march_opaque(hcol), qnh);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();   // G(s) and the faces of plane s in place; P free
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One tile's march: TJ x TK columns, or TK x TJ for a strip tile (tr); both
// shapes use the same LDS layout size.
template <int TJ, int TK, int LIM>
__device__ __forceinline__ void march_tile(double* lds, const BlockDesc& b, int tr, int j0, int k0, int pA,
                                           int pB, const double* __restrict__ qin, double* qout, int stage,
                                           const StageGas& gas, double dt) {
  static_assert(MarchGeom<TJ, TK>::NLDS == MarchGeom<TK, TJ>::NLDS, "transposed tile LDS");
  if constexpr (TJ == TK) {
    march_segment<TJ, TK, LIM>(lds, b, j0, k0, pA, pB, qin, b.q, qout, gas, dt, stage);
  } else {
    if (tr) march_segment<TK, TJ, LIM>(lds, b, j0, k0, pA, pB, qin, b.q, qout, gas, dt, stage);
    else march_segment<TJ, TK, LIM>(lds, b, j0, k0, pA, pB, qin, b.q, qout, gas, dt, stage);
  }
}

// Plain launch: grid = segments x march_tiling(...).count(), XCD-remapped.
// Segments split the block's planes evenly (lengths differ by at most one).
template <int TJ, int TK, int LIM, int WPE>
__global__ void __launch_bounds__(TJ * TK) __attribute__((amdgpu_waves_per_eu(WPE)))
k_stage_march(BlockDesc b, int stage, StageGas gas, double dt, int len) {
  __shared__ double lds[MarchGeom<TJ, TK>::NLDS];
  const int w = xcd_remap(blockIdx.x, gridDim.x);
  const MarchTiling mt = march_tiling(TJ, TK, b.nj, b.nk);
  const int nt = mt.count(), seg = w / nt;
  int j0, k0, tr;
  march_tile_of(mt, TJ, TK, w - seg * nt, j0, k0, tr);
  int pA, pB;
  march_segment_bounds(seg, march_nseg(b.ni, len), b.ni, pA, pB);
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  march_tile<TJ, TK, LIM>(lds, b, tr, j0, k0, pA, pB, qin, qout, stage, gas, dt);
}

// Batched launch over a tile table whose i0 is 2 x segment index + strip bit.
template <int TJ, int TK, int LIM, int WPE>
__global__ void __launch_bounds__(TJ * TK) __attribute__((amdgpu_waves_per_eu(WPE)))
k_stage_march_batched(const BlockDesc* __restrict__ blocks, const Tile3* __restrict__ tiles, int stage, StageGas gas,
                      double dt, int len) {
  __shared__ double lds[MarchGeom<TJ, TK>::NLDS];
  const Tile3 tl = tiles[xcd_remap(blockIdx.x, gridDim.x)];
  const BlockDesc& b = blocks[tl.block];
  int pA, pB;
  march_segment_bounds(tl.i0 >> 1, march_nseg(b.ni, len), b.ni, pA, pB);
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  march_tile<TJ, TK, LIM>(lds, b, tl.i0 & 1, tl.j0, tl.k0, pA, pB, qin, qout, stage, gas, dt);
}

}  // namespace famrdp

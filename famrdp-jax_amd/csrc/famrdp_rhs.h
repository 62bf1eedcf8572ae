// The two RHS terms on their own (rhs/invscd.py:53-131, rhs/viscous.py:30-108),
// for callers with an integrator of their own.
//
// Both work on tiles in LDS, so that a cell's primitives, a face's flux and a
// cell's viscous tensor are evaluated once: a thread per cell evaluated every
// flux twice and 15 cells' primitives for it, and the tensors went through a
// work array.  Indices are 64-bit and blocks of any size are taken.  The
// inviscid fluxes are the stage kernels' with every root, reciprocal and van
// Leer quotient rounded once; primitives, temperature, viscous tensors and the
// division by the volume are IEEE quotients, and the divergence takes the
// difference of two tensors before it takes the metrics, all as a thread per
// cell did.  Error against 80-bit arithmetic, rms over the largest value, 24 x
// 21 x 28 random cells (in brackets a thread per cell with IEEE quotients):
//   5 % noise    unit metrics  3.3e-16 (3.4e-16), viscous 3.6e-16 (3.6e-16)
//                curvilinear   1.2e-16 (1.3e-16), viscous 3.2e-16 (3.2e-16)
//   jumps of e^2 unit metrics  1.7e-17 (1.7e-17), viscous 1.2e-17 (1.2e-17)
//                curvilinear   1.4e-17 (1.3e-17), viscous 1.2e-17 (1.2e-17)
// With reciprocal roots and their squares the inviscid ones at jumps are
// 2.1e-17 and 1.6e-17; with the stage kernels' tensor and running divergence
// the viscous ones 1.3e-17.
#pragma once

namespace famrdp {

// Values computed by here, and nothing moved across.
struct PinFence {
  template <class... T>
  DF void operator()(T&... x) const {
    (march_pin(x), ...);
    __builtin_amdgcn_sched_barrier(0);
  }
};

// One tile at (i0, j0, k0).  FAST: fluxes by roe_flux2; *odd is set where one met
// a floor or is not finite.  Otherwise by the reference's own
// formulas (rhs/invscd.py:53-97): for tiles that hold the states a caller looks
// for (a density that is not positive, no pressure, NaN, infinities) or a face
// without area, where roe_flux2's identities and floors give other values.
template <int TI, int TJ, int TK, int LIM, bool FAST>
__device__ __forceinline__ void invscd_tile(double* s_pv, double* s_f, int* odd, const double* __restrict__ q,
                                            const double* __restrict__ kxyz, const double* __restrict__ vol,
                                            double* __restrict__ rhs, int ni, int nj, int nk, int i0, int j0, int k0,
                                            const StageGas& gas, double gamma) {
  EXACT_FP
  using C = CrossGeom<TI, TJ, TK>;
  using W = WideGeom<TI, TJ, TK>;
  const int64_t N = (int64_t)ni * nj * nk, si = (int64_t)nj * nk;
  const int t = opaque((int)threadIdx.x);   // slots are not held from tile to tile
  // ---- the face's metrics are on their way while the cells are staged ---------
  const int hf = t < C::NF ? t : C::NF - 1;
  const int D = W::face_axis_of(hf);
  const Loc3 l = W::face_cell(hf);
  const int ai = i0 + l.x, aj = j0 + l.y, ak = k0 + l.z;
  const int n_d = D == 0 ? ni : (D == 1 ? nj : nk);
  const int a = (D == 0 ? ai : (D == 1 ? aj : ak)) - 1;   // cell left of the face
  const bool ok = t < C::NF && ai < ni && aj < nj && ak < nk && a >= 1 && a <= n_d - 3;
  const int64_t cr = ok ? (int64_t)ai * si + (int64_t)aj * nk + ak : 0;
  const int64_t cl = ok ? cr - (D == 0 ? si : (D == 1 ? (int64_t)nk : (int64_t)1)) : 0;
  const double* kd = kxyz + 3 * D * N;
  double kl[3], kr[3];
  auto load_metrics = [&] {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      kl[m] = kd[m * N + cl];
      kr[m] = kd[m * N + cr];
    }
  };
  if constexpr (FAST) load_metrics();
  for (int h = t; h < C::NC; h += C::NTH) {
    const Loc3 s = C::cell(h);
    // no face reads a cell outside the block: any address in it will do there
    const int i = min(max(i0 + s.x, 0), ni - 1), j = min(max(j0 + s.y, 0), nj - 1), k = min(max(k0 + s.z, 0), nk - 1);
    const int64_t c = (int64_t)i * si + (int64_t)j * nk + k;
    double pv[5];
    load_prim(q, N, c, gamma, pv);
#pragma unroll
    for (int v = 0; v < 5; ++v) s_pv[v * C::NC + h] = pv[v];
  }
  __syncthreads();
  if (ok) {
    double F[5];
    if constexpr (FAST) {
      double p4[4][5];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int sl = C::step(l, D, s - 2);
#pragma unroll
        for (int v = 0; v < 5; ++v) p4[s][v] = s_pv[v * C::NC + sl];
      }
#pragma unroll
      for (int m = 0; m < 3; ++m) { kl[m] = 0.5 * kl[m]; kr[m] = 0.5 * kr[m]; }
      const bool plain = face_flux2<LIM, true>(p4[0], p4[1], p4[2], p4[3], kl, kr, gas, F);
      if (!(plain && isfinite(((F[0] + F[1]) + (F[2] + F[3])) + F[4]))) *odd = 1;
    } else {
      // (a variable at a time: the states of four cells at once take registers
      // that the fluxes of ordinary tiles would pay for)
      double pL[5], pR[5], U[2][5];
      int sl[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) sl[s] = C::step(l, D, s - 2);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double* p = s_pv + v * C::NC;
        const double d = p[sl[2]] - p[sl[1]];
        pL[v] = p[sl[1]] + 0.5 * limit(LIM, p[sl[1]] - p[sl[0]], d);
        pR[v] = p[sl[2]] - 0.5 * limit(LIM, d, p[sl[3]] - p[sl[2]]);
        march_pin(pL[v]);
        march_pin(pR[v]);
        __builtin_amdgcn_sched_barrier(0);
      }
      prim_to_cons(pL, gamma, U[0]);
      march_pin(U[0]);
      __builtin_amdgcn_sched_barrier(0);
      prim_to_cons(pR, gamma, U[1]);
      march_pin(U[1]);
      __builtin_amdgcn_sched_barrier(0);
      load_metrics();
      const double n[3] = {0.5 * (kl[0] + kr[0]), 0.5 * (kl[1] + kr[1]), 0.5 * (kl[2] + kr[2])};
      const double nm = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]) + 1e-300;
      double nu[3] = {n[0] / nm, n[1] / nm, n[2] / nm};
      march_pin(nu);
      __builtin_amdgcn_sched_barrier(0);
      roe_flux(U[0], U[1], nu, gamma, 0.1, F, PinFence{});
#pragma unroll
      for (int v = 0; v < 5; ++v) F[v] = 2.0 * (F[v] * nm);
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) s_f[v * C::NF + t] = F[v];
  }
  __syncthreads();
  for (int h = t; h < 5 * C::NT; h += C::NTH) {
    const int v = h / C::NT, o = h % C::NT, x = o / (TJ * TK), y = o / TK % TJ, z = o % TK;
    const int i = i0 + x, j = j0 + y, k = k0 + z;
    if (i >= ni || j >= nj || k >= nk) continue;
    const double* f = s_f + v * C::NF;
    double A = 0.0;
    bool any = false;
    auto axis = [&](int g, int n, int lo, int up) {
      if (g < 2 || g > n - 3) return;
      A = A + (f[lo + up] - f[lo]);
      any = true;
    };
    axis(i, ni, W::template low_face<0>(x, y, z), W::template high_face<0>());
    axis(j, nj, W::template low_face<1>(x, y, z), W::template high_face<1>());
    axis(k, nk, W::template low_face<2>(x, y, z), W::template high_face<2>());
    const int64_t c = (int64_t)i * si + (int64_t)j * nk + k;
    rhs[v * N + c] = any ? 0.0 - 0.5 * A / (vol[c] + 1e-300) : 0.0;
  }
  __syncthreads();
}

// -(F(c+1/2) - F(c-1/2)) / (vol + 1e-300) summed over the axes along which
// 2 <= c <= n-3, zero elsewhere.  A workgroup per tile, up to a limit of the
// grid beyond which they take several.  A thread per face of the tile, then a thread per
// variable and cell.  Tiles that hold an invalid state are done again afterwards,
// in registers that the first pass has anyway (PinFence): inside it, or without
// the fences, its spills cost every tile 10-20 %.  Bound by FP64 issue: 68 x 52
// x 84 cells 31.5 us in the trace (83.6 as a thread per cell), launches back to
// back 27.1, 132^3 196.  (With the stage kernels' six seeds a flux 28.6 in the
// trace, 132^3 207 there; the other tiles then 4x4x8 29.7 and 224, 3x4x4 31.4
// and 247, 2x4x8 29.4 and 225; six waves per SIMD, spills, 28.0 and 225.)
template <int TI, int TJ, int TK, int LIM>
__global__ void __launch_bounds__((CrossGeom<TI, TJ, TK>::NTH)) __attribute__((amdgpu_waves_per_eu(5)))
k_invscd_rhs(const double* __restrict__ q, const double* __restrict__ kxyz, const double* __restrict__ vol,
             double* __restrict__ rhs, int ni, int nj, int nk, StageGas gas, double gamma) {
  using C = CrossGeom<TI, TJ, TK>;
  __shared__ double s_pv[5 * C::NC];
  __shared__ double s_f[5 * C::NF];
  __shared__ int s_odd;                     // a flux of the tiles met a floor or is not finite
  // (a block that fits in memory has fewer than 2^31 tiles: 32-bit divisions)
  const unsigned ntj = (nj + TJ - 1) / TJ, ntk = (nk + TK - 1) / TK, ntile = (ni + TI - 1) / TI * ntj * ntk;
  const unsigned wg = xcd_remap(blockIdx.x, gridDim.x);
  if (threadIdx.x == 0) s_odd = 0;
  for (unsigned tile = wg; tile < ntile; tile += gridDim.x)
    invscd_tile<TI, TJ, TK, LIM, true>(s_pv, s_f, &s_odd, q, kxyz, vol, rhs, ni, nj, nk, tile / ntk / ntj * TI,
                                       tile / ntk % ntj * TJ, tile % ntk * TK, gas, gamma);
  if (__builtin_expect(__builtin_amdgcn_readfirstlane(s_odd) == 0, 1)) return;
  for (unsigned tile = wg; tile < ntile; tile += gridDim.x)
    invscd_tile<TI, TJ, TK, LIM, false>(s_pv, s_f, &s_odd, q, kxyz, vol, rhs, ni, nj, nk, tile / ntk / ntj * TI,
                                        tile / ntk % ntj * TJ, tile % ntk * TK, gas, gamma);
}

// (0, viscous divergence) with the reference's periodic roll at the padded
// edges.  Tiles as above; staged cells and tensors as in the fused stage kernel.
// Bound by latency (two workgroups a CU): 68 x 52 x 84 cells 26.9 us (tensors
// through memory 17.5 + 15.7), 132^3 179.  (With the stage kernels' tensor 25.5
// and 171; the other tiles then 4x4x8 26.8 and 189, 4x4x4 26.9 and 200, 8x8x8
// 29.6 and 202.)
template <int TI, int TJ, int TK>
__global__ void __launch_bounds__((WideGeom<TI, TJ, TK>::NGW)) __attribute__((amdgpu_waves_per_eu(4)))
k_viscous_rhs(const double* __restrict__ q, const double* __restrict__ kxyz, double* __restrict__ rhs, int ni, int nj,
              int nk, Gas gas) {
  EXACT_FP
  using T = FusedGeom<TI, TJ, TK>;
  using W = WideGeom<TI, TJ, TK>;
  static constexpr int NTH = W::NGW;     // a thread per tensor; the first NT hold the tile's cells
  __shared__ double s_u[4 * T::NPV];     // u, v, w, T
  __shared__ double s_g[9 * T::NG];
  const int64_t N = (int64_t)ni * nj * nk, si = (int64_t)nj * nk;
  const int ntj = (nj + TJ - 1) / TJ, ntk = (nk + TK - 1) / TK;
  const int64_t ntile = (int64_t)((ni + TI - 1) / TI) * ntj * ntk;
  const bool small = ni < WRAP_ONCE_MIN || nj < WRAP_ONCE_MIN || nk < WRAP_ONCE_MIN;
  for (int64_t tile = xcd_remap(blockIdx.x, gridDim.x); tile < ntile; tile += gridDim.x) {
    const int tk = (int)(tile % ntk), tj = (int)(tile / ntk % ntj), ti = (int)(tile / ntk / ntj);
    const int i0 = ti * TI, j0 = tj * TJ, k0 = tk * TK;
    const int t = opaque((int)threadIdx.x);   // slots are not held from tile to tile
    auto cell = [&](const Loc3& l) -> int64_t {
      const int i = i0 + l.x, j = j0 + l.y, k = k0 + l.z;
      if (small) return (int64_t)wrap_mod(i, ni) * si + (int64_t)wrap_mod(j, nj) * nk + wrap_mod(k, nk);
      return (int64_t)wrap_once(i, ni) * si + (int64_t)wrap_once(j, nj) * nk + wrap_once(k, nk);
    };
    // ---- the tensor's metrics are on their way while the cells are staged --------
    const Loc3 l = W::g_cell(t < T::NG ? t : T::NG - 1);
    const int64_t cg = cell(l);
    double kh[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) kh[m] = kxyz[m * N + cg];
#pragma unroll
    for (int h0 = 0; h0 < T::NPV; h0 += NTH) {
      const int h = h0 + t;
      const int64_t c = cell(W::pv_cell(h < T::NPV ? h : T::NPV - 1));
      double pv[5];
      load_prim(q, N, c, gas.gamma, pv);
      if (h < T::NPV) {
        s_u[h] = pv[1];
        s_u[T::NPV + h] = pv[2];
        s_u[2 * T::NPV + h] = pv[3];
        s_u[3 * T::NPV + h] = temperature(pv, gas.R);
      }
    }
    __syncthreads();
    if (t < T::NG) {
      double d[3][4], uvw[5], g9[9];
      const int s0 = ((l.x + 1) * T::B0J + l.y + 1) * T::B0K + l.z + 1;
#pragma unroll
      for (int s = 0; s < 3; ++s) uvw[s + 1] = s_u[s * T::NPV + s0];
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const int sp = W::pv_step(l, e, 1), sm = W::pv_step(l, e, -1);
#pragma unroll
        for (int s = 0; s < 4; ++s) d[e][s] = 0.5 * (s_u[s * T::NPV + sp] - s_u[s * T::NPV + sm]);
      }
      viscous_flux(uvw, s_u[3 * T::NPV + s0], d, kh, gas, g9);
#pragma unroll
      for (int m = 0; m < 9; ++m) s_g[m * T::NG + t] = g9[m];
    }
    __syncthreads();
    const int i = i0 + l.x, j = j0 + l.y, k = k0 + l.z;
    if (t < T::NT && i < ni && j < nj && k < nk) {
      int sp[3], sm[3];
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        sp[e] = W::g_step(l, e, 1);
        sm[e] = W::g_step(l, e, -1);
      }
      double vis[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        vis[r] = 0.0;
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          const double* Gc = s_g + gidx(r, m) * T::NG;
          const double di = 0.5 * (Gc[sp[0]] - Gc[sm[0]]), dj = 0.5 * (Gc[sp[1]] - Gc[sm[1]]),
                       dk = 0.5 * (Gc[sp[2]] - Gc[sm[2]]);
          vis[r] = vis[r] + fma(dk, kh[6 + m], fma(dj, kh[3 + m], di * kh[m]));
        }
      }
      const int64_t c = (int64_t)i * si + (int64_t)j * nk + k;
      rhs[c] = 0.0;
#pragma unroll
      for (int v = 0; v < 4; ++v) rhs[(v + 1) * N + c] = vis[v];
    }
    __syncthreads();
  }
}

template <int TI, int TJ, int TK>
inline unsigned rhs_grid(int ni, int nj, int nk) {
  const int64_t n = (int64_t)((ni + TI - 1) / TI) * ((nj + TJ - 1) / TJ) * ((nk + TK - 1) / TK);
  return (unsigned)std::min<int64_t>(n, 1 << 22);   // a grid holds fewer than 2^32 threads
}

}  // namespace famrdp

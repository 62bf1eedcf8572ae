// Wide stage kernel: one RK3 stage of a small TI x TJ x TK tile whose pieces
// of work each have threads of their own.
//
// The fused kernel gives a cell to a thread and takes the tile's work in
// turns: viscous tensors, divergence, then the faces of each axis, every one
// a pass and a remainder pass behind a barrier.  On a small block that chain
// is the stage's time: one wave per SIMD or less, eight dependent passes,
// 13.6 us for 20^3 cells, 13.5 for 36^3 (here 5.4 and 9.9; a launch is 2 of
// them).  Here the first waves hold the tile's viscous
// tensors, the others a face each, of all three axes; a thread's first loads
// are all issued at the start and the stage has three barriers:
//  1. primitives and temperature of the tile and its halo into LDS;
//  2. viscous tensors beside the faces of all axes, into LDS;
//  3. the cells' viscous divergence, by the first waves, into LDS beside the
//     face differences (j, k, then i, the fused kernel's order), by the others;
//  4. the Shu-Osher update.
// The same expressions on the same inputs in the same order as the fused
// kernel: the same bits.
#pragma once

namespace famrdp {

template <int TI, int TJ, int TK, int W>
__device__ __forceinline__ int wide_cell(const BlockDesc& b, int i0, int j0, int k0, const Loc3& l) {
  return tile_cell_rel<W>(l.x + 2, l.y + 2, l.z + 2, i0, j0, k0, b.ni, b.nj, b.nk);
}

template <int TI, int TJ, int TK>
__device__ __forceinline__ int wide_cell(const BlockDesc& b, int i0, int j0, int k0, const Loc3& l) {
  const int w = fused_wrap_mode<TI, TJ, TK>(b.wrap_mod, i0, j0, k0, b.ni, b.nj, b.nk);
  if (w == WRAP_MOD) return wide_cell<TI, TJ, TK, WRAP_MOD>(b, i0, j0, k0, l);
  if (w == WRAP_NONE) return wide_cell<TI, TJ, TK, WRAP_NONE>(b, i0, j0, k0, l);
  return wide_cell<TI, TJ, TK, WRAP_ONCE>(b, i0, j0, k0, l);
}

template <int TI, int TJ, int TK, int LIM>
__device__ __forceinline__ void stage_tile_wide(const BlockDesc& b, int i0, int j0, int k0,
                                                const double* __restrict__ qin, const double* q0, double* qout,
                                                const StageGas& gas, double dt, int stage) {
  EXACT_FP
  using T = FusedGeom<TI, TJ, TK>;
  using Wd = WideGeom<TI, TJ, TK>;
  __shared__ double lds[Wd::NLDS];
  double* s_pv = lds;                     // [5][NPV], then [NPV] temperature
  double* s_T = lds + 5 * T::NPV;
  double* s_g = lds + 6 * T::NPV;         // [9][NG]
  double* s_f = s_g + 9 * T::NG;          // [5][NF]
  double* s_v = lds;                      // [4][NT] viscous divergence, over the primitives
  const int t = threadIdx.x;
  const int64_t N = b.N;
  const int ni = __builtin_amdgcn_readfirstlane(b.ni), nj = __builtin_amdgcn_readfirstlane(b.nj),
            nk = __builtin_amdgcn_readfirstlane(b.nk);
  const unsigned n1 = (unsigned)N, nb = n1 * 8u;   // cells, and bytes between variables
  const __amdgpu_buffer_rsrc_t rq = march_rsrc(qin, 5 * N), rk = march_rsrc(b.kxyz, 9 * N);
  const bool faces = __builtin_amdgcn_readfirstlane(t >= Wd::NGW ? 1 : 0) != 0;   // uniform in a wave

  // ---- loads: the staged cells, then what the thread's own work needs -----------
  double qq[Wd::NIT][5];
#pragma unroll
  for (int it = 0; it < Wd::NIT; ++it) {
    const int h = t + it * Wd::NTH;
    const unsigned c = wide_cell<TI, TJ, TK>(b, i0, j0, k0, Wd::pv_cell(h < T::NPV ? h : T::NPV - 1));
#pragma unroll
    for (int v = 0; v < 5; ++v) qq[it][v] = ldx(rq, c, v * nb);
  }
  auto stage_prims = [&]() {
#pragma unroll
    for (int it = 0; it < Wd::NIT; ++it) {
      const int h = t + it * Wd::NTH;
      if (h < T::NPV) {
        double pp[6];
        prim_and_temp(qq[it], gas, pp);
#pragma unroll
        for (int v = 0; v < 5; ++v) s_pv[v * T::NPV + h] = pp[v];
        s_T[h] = pp[5];
      }
    }
  };

  if (faces) {
    // ---- one face -------------------------------------------------------------
    const int h = t - Wd::NGW;
    const int hc = h < Wd::NF ? h : Wd::NF - 1;
    const int D = Wd::face_axis_of(hc);
    const Loc3 l = Wd::face_cell(hc);
    const int ai = i0 + l.x, aj = j0 + l.y, ak = k0 + l.z;
    const int n_d = D == 0 ? ni : (D == 1 ? nj : nk);
    const int a = (D == 0 ? ai : (D == 1 ? aj : ak)) - 1;   // cell left of the face
    const bool ok = h < Wd::NF && ai < ni && aj < nj && ak < nk && a >= 1 && a <= n_d - 3;
    const int st = D == 0 ? nj * nk : (D == 1 ? nk : 1);
    const unsigned cr = ok ? (ai * nj + aj) * nk + ak : 0;
    const unsigned cl = ok ? cr - st : 0;
    double kl[3], kr[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      kl[m] = ldx(rk, cl + 3 * D * n1, m * nb);
      kr[m] = ldx(rk, cr + 3 * D * n1, m * nb);
    }
    stage_prims();
    __syncthreads();
    if (ok) {
      double p4[4][5];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int sl = Wd::pv_step(l, D, s - 2);
#pragma unroll
        for (int v = 0; v < 5; ++v) p4[s][v] = s_pv[v * T::NPV + sl];
      }
      double kl2[3], kr2[3], F[5];
#pragma unroll
      for (int m = 0; m < 3; ++m) { kl2[m] = 0.5 * kl[m]; kr2[m] = 0.5 * kr[m]; }
      face_flux2<LIM>(p4[0], p4[1], p4[2], p4[3], kl2, kr2, gas, F);
#pragma unroll
      for (int v = 0; v < 5; ++v) s_f[v * Wd::NF + h] = F[v];
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- the first NT of these threads update a cell each ------------------------
    const int x = h / (TJ * TK), y = (h / TK) % TJ, z = h % TK;
    const int gi = i0 + x, gj = j0 + y, gk = k0 + z;
    const bool own = h < T::NT && gi < ni && gj < nj && gk < nk;
    const unsigned c = own ? (gi * nj + gj) * nk + gk : 0;
    const __amdgpu_buffer_rsrc_t r0 = march_rsrc(q0, stage == 1 ? 0 : 5 * N);   // stage 1 takes no q0: loads give 0
    const double vol = ldx(march_rsrc(b.vol, N), c, 0);
    double qs[5], qq0[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      qs[v] = ldx(rq, c, v * nb);
      qq0[v] = ldx(r0, c, v * nb);
    }
    __syncthreads();
    double A[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    auto difference = [&](int lo, int up, int g, int n) {
      if (g >= 2 && g <= n - 3) {
#pragma unroll
        for (int v = 0; v < 5; ++v) A[v] = A[v] + (s_f[v * Wd::NF + lo + up] - s_f[v * Wd::NF + lo]);
      }
    };
    if (own) {
      difference(Wd::template low_face<1>(x, y, z), Wd::template high_face<1>(), gj, nj);
      difference(Wd::template low_face<2>(x, y, z), Wd::template high_face<2>(), gk, nk);
      difference(Wd::template low_face<0>(x, y, z), Wd::template high_face<0>(), gi, ni);
    }
    const double rvh = 0.5 * rcp(vol + 1e-300);
    __syncthreads();
    if (!own) return;
    const StageCoef sc = stage_coef(stage, dt * b.dt_scale);
#pragma unroll
    for (int v = 0; v < 5; ++v)
      stx(march_rsrc(qout, 5 * N), c, v * nb,
          stage_update(sc, qq0[v], qs[v], A[v], rvh, v == 0 ? 0.0 : s_v[(v - 1) * T::NT + h]));
    return;
  }

  // ---- one viscous tensor; the first NT of these threads hold the tile's cells --
  const Loc3 l = Wd::g_cell(t < T::NG ? t : T::NG - 1);
  const unsigned c = wide_cell<TI, TJ, TK>(b, i0, j0, k0, l);
  double kh[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) kh[m] = ldx(rk, c, m * nb);
  const double cmu = uniform(gas.cmu * b.mu0);
  stage_prims();
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 9; ++m) kh[m] = 0.5 * kh[m];
  if (t < T::NG) {
    const int s0 = ((l.x + 1) * T::B0J + l.y + 1) * T::B0K + l.z + 1;   // a tensor's cell lies in the box
    const double uvwT[4] = {s_pv[T::NPV + s0], s_pv[2 * T::NPV + s0], s_pv[3 * T::NPV + s0], s_T[s0]};
    double d[3][4];
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int sp = Wd::pv_step(l, e, 1), sm = Wd::pv_step(l, e, -1);
      d[e][0] = s_pv[T::NPV + sp] - s_pv[T::NPV + sm];
      d[e][1] = s_pv[2 * T::NPV + sp] - s_pv[2 * T::NPV + sm];
      d[e][2] = s_pv[3 * T::NPV + sp] - s_pv[3 * T::NPV + sm];
      d[e][3] = s_T[sp] - s_T[sm];
    }
    double g9[9];
    viscous_flux_fast(uvwT, d, kh, cmu, gas, g9);
#pragma unroll
    for (int m = 0; m < 9; ++m) s_g[m * T::NG + t] = g9[m];
  }
  __syncthreads();

  // ---- viscous divergence of the tile's cells ------------------------------------
  if (t < T::NT) {
    double vis[4] = {0.0, 0.0, 0.0, 0.0};
    const int sp[3] = {Wd::g_step(l, 0, 1), Wd::g_step(l, 1, 1), Wd::g_step(l, 2, 1)};
    const int sm[3] = {Wd::g_step(l, 0, -1), Wd::g_step(l, 1, -1), Wd::g_step(l, 2, -1)};
    double gi[9], dj[9], dk[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) gi[m] = s_g[m * T::NG + sm[0]];
    visc_div_im(gi, kh, vis);
    march_pin(vis);   // here, not sunk to the update: few tensors at a time in registers
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      const double* Gc = s_g + m * T::NG;
      dj[m] = Gc[sp[1]] - Gc[sm[1]];
      dk[m] = Gc[sp[2]] - Gc[sm[2]];
    }
    visc_div_jk(dj, dk, kh, vis);
    march_pin(vis);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 9; ++m) gi[m] = s_g[m * T::NG + sp[0]];
    visc_div_ip(gi, kh, vis);
    march_pin(vis);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < 4; ++v) s_v[v * T::NT + t] = vis[v];
  }
  __syncthreads();
}

// Six waves per SIMD (80 registers, six of them spilled for 3x4x4): its
// workgroups of five waves then pack four to a CU whatever SIMDs their waves
// land on (at five waves and no spill 36^3 takes 10.8 us instead of 9.8, 72^3
// 60.4 instead of 56.6).
template <int TI, int TJ, int TK, int LIM>
__global__ void __launch_bounds__((WideGeom<TI, TJ, TK>::NTH)) __attribute__((amdgpu_waves_per_eu(6)))
k_stage_wide(BlockDesc b, int stage, StageGas gas, double dt, int ntj, int ntk) {
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int tk = t % ntk, tj = (t / ntk) % ntj, ti = t / (ntk * ntj);
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  stage_tile_wide<TI, TJ, TK, LIM>(b, ti * TI, tj * TJ, tk * TK, qin, b.q, qout, gas, dt, stage);
}

template <int TI, int TJ, int TK, int LIM>
__global__ void __launch_bounds__((WideGeom<TI, TJ, TK>::NTH)) __attribute__((amdgpu_waves_per_eu(6)))
k_stage_wide_batched(const BlockDesc* __restrict__ blocks, const Tile3* __restrict__ tiles, int stage, StageGas gas,
                     double dt) {
  const Tile3 tl = tiles[xcd_remap(blockIdx.x, gridDim.x)];
  const BlockDesc& b = blocks[tl.block];
  const double* qin = stage == 1 ? b.q : (stage == 2 ? b.q1 : b.q2);
  double* qout = stage == 1 ? b.q1 : (stage == 2 ? b.q2 : b.q);
  stage_tile_wide<TI, TJ, TK, LIM>(b, tl.i0, tl.j0, tl.k0, qin, b.q, qout, gas, dt, stage);
}

}  // namespace famrdp

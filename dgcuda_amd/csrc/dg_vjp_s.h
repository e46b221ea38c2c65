// dg_vjp_s.h -- the right-hand side's vector-Jacobian product on small
// meshes: a thread per point, then a thread per coefficient, as the small
// mesh stage (dg_stage_s.h).  For Maxwell TE's permittivity gradient, whose
// impedance terms are a launch of their own on the wide path (k_eps_side), the
// side points form those terms too.
// Included by dg_adjoint.hip (the flux VJPs it uses are defined there).
#pragma once

#include "dg_stage_s.h"

namespace dgk {

template <int PHYS, int P, bool EPS, bool FULL>
__global__ __launch_bounds__((small_t<PHYS, P, FULL, true>())) void k_vjp_s(const AdjArgs a) {
  using TC = TabC<P>;
  constexpr int NP = TC::NP, NQ = TC::NQ, NQ1 = TC::NQ1, N = nvars_of(PHYS);
  constexpr bool TE = PHYS == PH_TE;
  constexpr bool kU = EPS || !linear_flux<PHYS>();  // the state is read
  constexpr int EB = small_eb(P), NR = N * NP, NS = 3 * NQ1, T = small_t<PHYS, P, FULL, true>();
  constexpr int RW = T / EB, R = (NR + RW - 1) / RW, RN = (3 * NR + RW - 1) / RW;
  constexpr int NV = small_nv<PHYS>(), NPU = kU ? NP : 1;
  __shared__ double s_B[NP * NQ], s_side[3 * NP * NQ1];
  __shared__ dbl2 s_G[NP * NQ];
  __shared__ __align__(16) double s_w[NP][EB][NV], s_nw[3][NP][EB][NV];
  __shared__ __align__(16) double s_u[NPU][EB][NV], s_nu[3][NPU][EB][NV];
  __shared__ __align__(16) double s_f[NS][EB][NV], s_g[NQ][EB][NV];
  __shared__ double s_z[EPS ? NS : 1][EB], s_k[EPS ? 2 * NP : 1][EB];
  const int t = threadIdx.x, el = t % EB, row = t / EB;
  const int K = a.m.K;
  const int e = remap_block(blockIdx.x, (K + EB - 1) / EB) * EB + el;
  const bool act = e < K;
  const int ee = act ? e : K - 1;

  // ---- loads
  int nbq[RN];
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW, rr = r < 3 * NR ? r : 0;
    nbq[q] = a.m.slot[(size_t)(rr / NR) * K + ee].x;
  }
  constexpr int SV = small_side_t<P, FULL>();  // the first volume point's thread
  const bool is_side = t < EB * NS, is_vol = t >= SV && t < SV + EB * NQ;
  const int sp = is_side ? row : 0, sk = sp / NQ1, jj = sp - sk * NQ1;
  const int vj = is_vol ? row - SV / EB : 0;
  const int2 sl = a.m.slot[(size_t)sk * K + ee];
  double ow[R], ou[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW, rr = r < NR ? r : 0;
    ow[q] = gld(a.lam + (size_t)rr * K, ee);
    ou[q] = 0.;
    if constexpr (kU) ou[q] = gld(a.us + (size_t)rr * K, ee);
  }
  const double xr = gld(a.m.xr, ee), yr = gld(a.m.yr, ee);
  const double xs = gld(a.m.xs, ee), ys = gld(a.m.ys, ee);
  const double Jme = gld(a.m.J, ee);
  double eps_me = 1., eps_nb = 1.;
  if constexpr (TE) eps_me = gld(a.m.eps, ee);
  double Vv[6] = {0., 0., 0., 0., 0., 0.};
  const bool vary = PHYS == PH_ADV && a.ph.prob == PB_ADV_ROTHILL;
  if (vary) {
#pragma unroll
    for (int q = 0; q < 6; q++) Vv[q] = gld(a.m.V + (size_t)q * K, ee);
  }
  for (int q = t; q < NP * NQ; q += T) {
    s_B[q] = TC::B[q];
    s_G[q] = dbl2{TC::GX[q], TC::GY[q]};
  }
  for (int q = t; q < 3 * NP * NQ1; q += T) s_side[q] = TC::SIDE[q];
  // the neighbours and this point's side, no branch between the loads (as the
  // stage's)
  const int sid = sl.y >> 3;
  double nw[RN], nu[RN];
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW, nr = r < 3 * NR ? r % NR : 0, nb = nbq[q] >= 0 ? nbq[q] : ee;
    nw[q] = gld(a.lam + (size_t)nr * K, nb);
    nu[q] = 0.;
    if constexpr (kU) nu[q] = gld(a.us + (size_t)nr * K, nb);
  }
  double nx = 0., ny = 0., len = 0., Jnb = 1., bv[NMAX] = {0., 0., 0., 0.};
  if (is_side) {
    nx = gld(a.m.snx, sid);
    ny = gld(a.m.sny, sid);
    len = gld(a.m.slen, sid);
    const int snb_e = sl.x >= 0 ? sl.x : ee, bslot = a.m.side[sid].w;
    Jnb = gld(a.m.J, snb_e);
    if constexpr (TE) eps_nb = gld(a.m.eps, snb_e);
    if (sl.x < 0) {
      const double *b = a.m.bnd_val + ((size_t)bslot * NQ1 + jj) * NMAX;
#pragma unroll
      for (int n = 0; n < NMAX; n++) bv[n] = b[n];
    }
  }
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW, nr = r % NR;
    const bool has = nbq[q] >= 0;
    if (r < 3 * NR) {
      s_nw[r / NR][nr % NP][el][nr / NP] = has ? nw[q] : 0.;
      if constexpr (kU) s_nu[r / NR][nr % NP][el][nr / NP] = has ? nu[q] : 0.;
    }
  }
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW;
    if (r < NR) {
      s_w[r % NP][el][r / NP] = ow[q];
      if constexpr (kU) s_u[r % NP][el][r / NP] = ou[q];
    }
  }
  // the weights' scale dt / J (TE also 1/eps, 1/mu per row), times lc
  const double sme = a.lc * (a.dt / Jme);
  auto scale = [&](double s, double eps, int n) {
    if constexpr (TE) return s * (n < 2 ? 1. / eps : 1. / a.ph.mu);
    return s;
  };
  __syncthreads();

  // ---- points
  if (is_side) {
    const int nb = sl.x, nbls = sl.y & 3, role = (sl.y >> 2) & 1;
    const double *po = s_side + (size_t)(sk * NP) * NQ1 + jj;
    const double *pn = s_side + (size_t)(nbls * NP) * NQ1 + NQ1 - 1 - jj;
    double Um[NMAX] = {0., 0., 0., 0.}, Un[NMAX] = {0., 0., 0., 0.}, Wm[N], Wn[N];
#pragma unroll
    for (int n = 0; n < N; n++) Wm[n] = Wn[n] = 0.;
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const double x = po[i * NQ1], y = pn[i * NQ1];
      double wm[N], wn[N], um[N], un[N];
      lds_get<N>(s_w[i][el], wm);
      lds_get<N>(s_nw[sk][i][el], wn);
      if constexpr (kU) {
        lds_get<N>(s_u[i][el], um);
        lds_get<N>(s_nu[sk][i][el], un);
      }
#pragma unroll
      for (int n = 0; n < N; n++) {
        Wm[n] = fma(wm[n], x, Wm[n]);
        Wn[n] = fma(wn[n], y, Wn[n]);
        if constexpr (kU) {
          Um[n] = fma(um[n], x, Um[n]);
          Un[n] = fma(un[n], y, Un[n]);
        }
      }
    }
    if constexpr (kU) {
      if (nb == -1) {
        wall_state<PHYS>(a.ph, Um, Un, bv[0], bv[1], bv[2]);
      } else if (nb < 0) {
#pragma unroll
        for (int n = 0; n < N; n++) Un[n] = bv[n];
      }
    }
    const double snb = a.lc * (a.dt / Jnb);
    const double f = (role ? 0.5 : -0.5) * len * TC::W1[jj];
    double UL[NMAX], UR[NMAX], gF[NMAX] = {0., 0., 0., 0.}, gL[NMAX] = {0., 0., 0., 0.},
                               gR[NMAX] = {0., 0., 0., 0.};
#pragma unroll
    for (int n = 0; n < NMAX; n++) {
      UL[n] = role ? Un[n] : Um[n];
      UR[n] = role ? Um[n] : Un[n];
    }
#pragma unroll
    for (int n = 0; n < N; n++)
      gF[n] = f * (scale(sme, eps_me, n) * Wm[n] - scale(snb, eps_nb, n) * Wn[n]);
    PhysParams pv = a.ph;
    if constexpr (PHYS == PH_ADV) {
      if (vary) {
        double x, y;
        side_point<NQ1>(Vv, TC::X1, sk, jj, x, y);
        rothill_velocity(x, y, pv.ax, pv.ay);
      }
    }
    double gzl, gzr;
    riemann_vjp<PHYS>(pv, UL, UR, nx, ny, role ? eps_nb : eps_me, role ? eps_me : eps_nb, gF, gL,
                      gR, gzl, gzr);
    double gme[NMAX];
#pragma unroll
    for (int n = 0; n < N; n++) gme[n] = role ? gR[n] : gL[n];
    if (nb == -1) wall_vjp<PHYS>(a.ph, bv[0], bv[1], bv[2], gR, gme);
    lds_put<N>(s_f[sp][el], gme);
    // a boundary's ghost state carries the element's own impedance
    if constexpr (EPS) s_z[sp][el] = nb < 0 ? gzl + gzr : (role ? gzr : gzl);
  } else if (is_vol) {
    double U[NMAX] = {0., 0., 0., 0.}, gfx[NMAX], gfy[NMAX], gU[NMAX] = {0., 0., 0., 0.};
    double wa[N], wb[N];
#pragma unroll
    for (int n = 0; n < N; n++) wa[n] = wb[n] = 0.;
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const dbl2 G = s_G[i * NQ + vj];
      double wm[N], um[N];
      lds_get<N>(s_w[i][el], wm);
      if constexpr (kU) lds_get<N>(s_u[i][el], um);
#pragma unroll
      for (int n = 0; n < N; n++) {
        wa[n] = fma(wm[n], G.x, wa[n]);
        wb[n] = fma(wm[n], G.y, wb[n]);
        if constexpr (kU) U[n] = fma(um[n], s_B[i * NQ + vj], U[n]);
      }
    }
#pragma unroll
    for (int n = 0; n < N; n++) {
      const double sc = scale(sme, eps_me, n);
      gfx[n] = sc * (wa[n] * ys - wb[n] * yr);
      gfy[n] = sc * (wb[n] * xr - wa[n] * xs);
    }
    PhysParams pv = a.ph;
    if constexpr (PHYS == PH_ADV) {
      if (vary) {
        double x, y;
        elem_point(Vv, TC::R1[vj], TC::R2[vj], x, y);
        rothill_velocity(x, y, pv.ax, pv.ay);
      }
    }
    fn_vjp<PHYS>(pv, U, 1.0, 0.0, gfx, gU);
    fn_vjp<PHYS>(pv, U, 0.0, 1.0, gfy, gU);
    lds_put<N>(s_g[vj][el], gU);
  }
  __syncthreads();

  // ---- modes
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW;
    if (r < NR) {
      const int n = r / NP, i = r % NP;
      const size_t o = (size_t)r * K;
      // the combination arrays first: they are in flight during the sums
      double x[4];
#pragma unroll
      for (int u = 0; u < 4; u++) x[u] = u < a.nout ? gld(a.ot[u] + o, ee) : 0.;
      double g = 0.;
#pragma unroll
      for (int j = 0; j < NQ; j++) g = fma(s_g[j][el][n], s_B[i * NQ + j], g);
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < NQ1; j++)
          g = fma(s_f[k * NQ1 + j][el][n], s_side[(k * NP + i) * NQ1 + j], g);
      double v = a.scale * g;
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (u < a.nout) v = fma(a.oc[u], x[u], v);
      if (act) gst(a.gout + o, e, v);
      if constexpr (EPS) {
        if (n < 2) s_k[r][el] = ow[q] * gld(a.kst + o, ee);
      }
    }
  }
  if constexpr (EPS) {
    __syncthreads();
    if (row == 0 && act) {
      // dz/deps = -z / (2 eps) on the sides, and the row scaling
      // -lc lam . k_E / eps
      double gz = 0., ew = 0.;
      for (int s = 0; s < NS; s++) gz += s_z[s][el];
      for (int r = 0; r < 2 * NP; r++) ew += s_k[r][el];
      const double z = sqrt(a.ph.mu / eps_me);
      a.geps[e] += gz * (-z / (2. * eps_me)) - a.lc * ew / eps_me;
    }
  }
}

}  // namespace dgk

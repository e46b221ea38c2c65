// dg_limit.h -- the p = 1 slope limiter inside a Runge-Kutta stage.
//
// The reference limits every stage's k = dt L(u) and the step's result
// (limit_c conserv_kernels.cu:640-720), each of which needs the finished means
// of the three neighbours.  A limited stage is therefore two launches: the
// stage kernel stores the plain k, and k_limited limits it, forms the stage
// combination, applies the element-local positivity fix to what the next stage
// reads, and after the last stage limits the combined state too: the limiter
// keeps means, so a neighbour's new mean follows from rows 0 of what the
// combination reads and no finished state is waited for.  The result goes to
// another buffer than the step base, whose neighbour means are read here.
// Bound by latency (a launch and two dependent memory round trips): a thread
// per (element, variable), 16 elements per one-wave block on small meshes so
// that a few thousand elements reach every CU, 64 (full lines per row) above.
// us per RK4 stage (Euler, periodic mesh, step close included), with the
// limiter, the combinations, the fix and the CFL pass as launches of their own
// before, and now: 1,058 triangles 24.1 / 11.0, 11,250 26.4 / 11.1, 12,800
// 26.1 / 12.0, 131,072 40.2 / 28.3, 524,288 113.5 / 89.6.
#pragma once

#include "dg_stage_s.h"

namespace dgk {

// the limiter's factor of a variable's two linear modes (limit_c :660-716).
// The reference's minimum over the six side points of (Uc - Umin) / (Ui - Uc)
// for Ui > Uc, and of its counterpart below, is one division each by the
// largest difference: the numerators do not depend on the point and a rounded
// quotient is monotone in its divisor.
__device__ __forceinline__ double limit_factor(double c0, double c1, double c2, const double *m) {
  using TC = TabC<1>;
  const double Uc = c0 * TC::B[0];
  double Umin = Uc, Umax = Uc, up = 0., dn = 0.;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double Ui = m[k] * TC::B[0];
    Umin = Ui < Umin ? Ui : Umin;
    Umax = Ui > Umax ? Ui : Umax;
  }
#pragma unroll
  for (int s = 0; s < 3; s++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      double Ui = 0.;
      Ui += c0 * TC::SIDE[(s * 3 + 0) * 2 + j];
      Ui += c1 * TC::SIDE[(s * 3 + 1) * 2 + j];
      Ui += c2 * TC::SIDE[(s * 3 + 2) * 2 + j];
      if (Ui > Uc) up = fmax(up, Ui - Uc);
      if (Ui < Uc) dn = fmin(dn, Ui - Uc);
    }
  double a = 1.;
  if (up > 0.) a = fmin(a, (Uc - Umin) / up);
  if (dn < 0.) a = fmin(a, (Uc - Umax) / dn);
  return a < 0. ? 0. : a;
}

constexpr int limited_threads(int n, int eb) { return (n * eb + 63) / 64 * 64; }

template <int PHYS, int EB>
__global__ __launch_bounds__((limited_threads(nvars_of(PHYS), EB))) void k_limited(
    const LimArgs a) {
  constexpr int N = nvars_of(PHYS), T = limited_threads(N, EB), kW = T / 64;
  using TC = TabC<1>;
  __shared__ double s_c[3 * N][EB];
  __shared__ unsigned long long s_l[kW], s_k[kW];
  const int t = threadIdx.x, el = t % EB, row = t / EB, n = row < N ? row : 0;
  const int K = a.m.K;
  const int e = remap_block(blockIdx.x, a.nblk) * EB + el;
  const bool act = e < K, mine = act && row < N;
  const int ee = act ? e : K - 1;
  const size_t r0 = (size_t)(3 * n) * K;
  const bool stop = (a.st->nan_flag | a.st->halt) != 0;
  if (stop && !a.final) return;
  int nb[3];
#pragma unroll
  for (int k = 0; k < 3; k++) nb[k] = a.m.slot[(size_t)k * K + ee].x;
  const bool use_us = a.mode == M_A_UN_B_US_CK;
  const bool use_acc = a.accmode == ACC_ADD3 || a.accmode == ACC_FINAL6;
  double kk[3], un[3], us[3], ac[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const size_t r = r0 + (size_t)i * K;
    kk[i] = gld(a.k + r, ee);
    un[i] = gld(a.un + r, ee);
    us[i] = use_us ? gld(a.us + r, ee) : 0.;
    ac[i] = use_acc ? gld(a.acc + r, ee) : 0.;
  }
  if (stop) {  // a stopped run's state goes on unchanged
#pragma unroll
    for (int i = 0; i < 3; i++)
      if (mine) gst(a.out + r0 + (size_t)i * K, e, un[i]);
    return;
  }
  const double base[3] = {un[0], un[1], un[2]};
  if constexpr (has_positivity<PHYS>()) {
    if (a.fix && gld_int(a.bad, ee)) un[1] = un[2] = 0.;
  }
  // the neighbours' means (a boundary side: the element's own)
  double mk[3], mn[3], ms[3], ma[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int q = nb[k] < 0 ? ee : nb[k];
    mk[k] = gld(a.k + r0, q);
    mn[k] = ms[k] = ma[k] = 0.;
    if (a.final) {
      mn[k] = gld(a.un + r0, q);
      if (use_us) ms[k] = gld(a.us + r0, q);
      if (use_acc) ma[k] = gld(a.acc + r0, q);
    }
  }
  double f = limit_factor(kk[0], kk[1], kk[2], mk);
  kk[1] *= f;
  kk[2] *= f;
  // (time_integrator.cu:107-130)
  auto combine = [&](double u, double s, double c, double k) {
    if (a.accmode == ACC_FINAL6) return u + (c + k / 6.);
    if (use_us) return (a.A * u + a.B * s) + a.C * k;
    return u + a.C * k;
  };
  double o[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const size_t r = r0 + (size_t)i * K;
    if (mine && a.accmode == ACC_SET6) gst(a.acc + r, e, kk[i] / 6.);
    if (mine && a.accmode == ACC_ADD3) gst(a.acc + r, e, ac[i] + kk[i] / 3.);
    o[i] = combine(un[i], us[i], ac[i], kk[i]);
  }
  if (a.final) {
    double m[3];
#pragma unroll
    for (int k = 0; k < 3; k++) m[k] = combine(mn[k], ms[k], ma[k], mk[k]);
    f = limit_factor(o[0], o[1], o[2], m);
    o[1] *= f;
    o[2] *= f;
  }
  bool bad = false;
  if ((has_positivity<PHYS>() && a.fix) || a.final) {
    if (row < N) {
#pragma unroll
      for (int i = 0; i < 3; i++) s_c[3 * n + i][el] = o[i];
    }
    __syncthreads();
  }
  if constexpr (has_positivity<PHYS>()) {
    if (a.fix) {
      // every thread of the element comes to the same decision
      double u[N][3];
#pragma unroll
      for (int v = 0; v < N; v++)
#pragma unroll
        for (int i = 0; i < 3; i++) u[v][i] = s_c[3 * v + i][el];
      bad = needs_fix<PHYS, 1>(a.ph, u);
      if (a.final) {  // the state stays as computed; its readers take the flag
        if (act && row == 0) a.bad[e] = bad ? 1 : 0;
      } else if (bad) {
        o[1] = o[2] = 0.;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 3; i++)
    if (mine) gst(a.out + r0 + (size_t)i * K, e, o[i]);
  if (!a.final) return;
  // the step's maxima: the CFL speed and the change of rows r < N
  double lam = 0., dc = 0.;
  if (act && row == 0) {
    double U[NMAX];
#pragma unroll
    for (int v = 0; v < N; v++) U[v] = s_c[3 * v][el] * TC::B[0];
    PhysParams pv = a.ph;
    if constexpr (PHYS == PH_ADV) {
      if (a.ph.prob == PB_ADV_ROTHILL) {
        double V[6], x, y;
#pragma unroll
        for (int q = 0; q < 6; q++) V[q] = gld(a.m.V + (size_t)q * K, e);
        elem_point(V, TC::R1[TC::NQ / 2], TC::R2[TC::NQ / 2], x, y);
        rothill_velocity(x, y, pv.ax, pv.ay);
      }
    }
    lam = ref_max_operand(cfl_speed<PHYS>(pv, U, PHYS == PH_TE ? gld(a.m.eps, e) : 1.), e);
  }
  if (mine && a.conv) {
#pragma unroll
    for (int i = 0; i < 3; i++)
      if (3 * n + i < N) dc = fmax(dc, fabs(o[i] - base[i]));
  }
  unsigned long long kl = wave_max_key(ord_key(lam)), kc = wave_max_key(ord_key(dc));
  if ((t & 63) == 0) {
    s_l[t >> 6] = kl;
    s_k[t >> 6] = kc;
  }
  __syncthreads();
  if (t == 0) {
#pragma unroll
    for (int w = 1; w < kW; w++) {
      kl = s_l[w] > kl ? s_l[w] : kl;
      kc = s_k[w] > kc ? s_k[w] : kc;
    }
    a.part[blockIdx.x] = kl;
    if (a.conv) a.part[a.nblk + blockIdx.x] = kc;
  }
}

}  // namespace dgk

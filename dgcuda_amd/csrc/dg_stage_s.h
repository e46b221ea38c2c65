// dg_stage_s.h -- the RK stage on small meshes: a thread per point, then a
// thread per coefficient.
//
// On a mesh of a few thousand elements the one-thread-per-element stage is a
// single wave on a few CUs that walks tens of kilobytes of straight-line code
// (every table entry an immediate), so its time is the instruction stream of
// one wave and the chip idles.  Here a block of 256 threads takes EB elements:
//   load     the elements' own and their neighbours' coefficients into LDS,
//            with every other operand (tables, metric, step base) in flight
//   points   a thread per side or volume point: the states there, the
//            numerical or the contravariant flux, its components into LDS
//   modes    a thread per (variable, mode): the projection of the point
//            fluxes in the one-thread kernel's order, dt/J, the RK
//            combination, the store
// The tables are in LDS, so the code is a few kilobytes.  The same launch
// also does what the large-mesh path leaves to launches of their own: the
// first stage of a step closes the step before it (every block reduces the
// partials, block 0 stores the new step state), and time-dependent boundary
// data are evaluated by the side points that use them.
// Bound by latency (launch, two dependent memory round trips, LDS): rotating
// hill p = 4 on 1,080 triangles 26.4 us per RK4 stage with its boundary and
// close before, 6.6 us now; supersonic vortex p = 3 on 2,880 triangles 22.9 ->
// 10.0 us (fewer elements per block fill more CUs, but below the widths here
// the loads fall under 32 B per row).
#pragma once

#include "dg_stage.h"

namespace dgk {

// elements per block: the points (3 (p+1) side and n_q volume points each)
// of EB elements fit the block's 256 threads
__host__ __device__ constexpr int small_eb(int p) {
  return p == 0 ? 64 : p <= 2 ? 16 : p <= 4 ? 8 : 4;
}
constexpr int kSmallT = 256;

// needs_fix of the block's elements' new coefficients s_c (element-local
// positivity): rows 0 .. N-1 bound one variable each and every thread of an
// element takes the same decision from the bounds; where they do not settle
// it (rare), each thread checks one of its element's points
template <int PHYS, int P, int EB>
__device__ __forceinline__ bool small_needs_fix(const PhysParams &ph, const double (*s_c)[EB],
                                                const double *s_B, const double *s_side,
                                                double (*s_md)[nvars_of(PHYS)][EB], int *s_bad,
                                                int el, int row) {
  using TC = TabC<P>;
  constexpr int NP = TC::NP, NQ = TC::NQ, NQ1 = TC::NQ1, N = nvars_of(PHYS);
  constexpr double margin = 1e-10;
  if (row < N) {
    double d = 0.;
#pragma unroll
    for (int i = 1; i < NP; i++) d = fma(fabs(s_c[row * NP + i][el]), phi_bound<P>(i), d);
    s_md[0][row][el] = s_c[row * NP][el] * TC::B[0];
    s_md[1][row][el] = d * (1. + margin);
  }
  if (row == 0) s_bad[el] = 0;
  __syncthreads();
  double mean[N], dev[N];
#pragma unroll
  for (int n = 0; n < N; n++) {
    mean[n] = s_md[0][n][el];
    dev[n] = s_md[1][n][el];
  }
  const bool sure = bounds_physical<PHYS>(mean, dev);
  if (!__syncthreads_or(sure ? 0 : 1)) return false;
  if (!sure && row < NQ + 3 * NQ1) {
    const int sp = row - NQ;
    const double *t = sp < 0 ? s_B + row : s_side + sp / NQ1 * NP * NQ1 + sp % NQ1;
    const int st = sp < 0 ? NQ : NQ1;
    double U[NMAX];
#pragma unroll
    for (int n = 0; n < N; n++) U[n] = 0.;
#pragma unroll 1
    for (int i = 0; i < NP; i++)
#pragma unroll
      for (int n = 0; n < N; n++) U[n] = fma(s_c[n * NP + i][el], t[i * st], U[n]);
    if (!is_physical<PHYS>(ph, U)) s_bad[el] = 1;  // (every writer stores the same value)
  }
  __syncthreads();
  return s_bad[el] != 0;
}

// the problems whose outside states depend on time (the caller's boundary
// states and every wall do not): only their systems have the TDB form
template <int PHYS>
__host__ __device__ constexpr bool small_tdb() {
  return PHYS == PH_ADV || PHYS == PH_EULER;
}

// The step state of a small-mesh run has two slots: slot 0 is the state
// between steps (pending: a step was taken whose maxima wait in the
// partials), slot 1 the running step's.  The first stage reads slot 0,
// closes the pending step and stores slot 1; the later stages read slot 1;
// the last one stores it back to slot 0 as pending.  No launch reads a slot
// that it writes.
template <int PHYS, int P, bool TDB>
__global__ __launch_bounds__(kSmallT) void k_stage_s(const StageArgs a) {
  using TC = TabC<P>;
  constexpr int NP = TC::NP, NQ = TC::NQ, NQ1 = TC::NQ1, N = nvars_of(PHYS);
  constexpr int EB = small_eb(P), NR = N * NP, NS = 3 * NQ1, T = kSmallT;
  constexpr int RW = T / EB;                 // rows of one pass over the elements
  constexpr int R = (NR + RW - 1) / RW;      // passes over the own rows
  constexpr int RN = (3 * NR + RW - 1) / RW;  // and over the neighbours'
  static_assert(EB * (NS + NQ) <= T, "a thread per point");
  __shared__ double s_B[NP * NQ], s_GX[NP * NQ], s_GY[NP * NQ], s_side[3 * NP * NQ1];
  __shared__ double s_c[NR][EB], s_n[3 * NR][EB];
  __shared__ double s_f[NS][N][EB], s_g[NQ][2][N][EB];
  __shared__ double s_md[2][N][EB];
  __shared__ int s_bad[EB];
  __shared__ unsigned long long s_l[T / 64], s_k[T / 64];
  const int t = threadIdx.x, el = t % EB, row = t / EB;
  const int K = a.m.K;
  const int e = remap_block(blockIdx.x, a.nblk) * EB + el;
  const bool act = e < K;
  const int ee = act ? e : K - 1;
  const bool use_un = a.accmode == ACC_FINAL6 || a.mode == M_A_UN_B_US_CK || a.mode == M_UN_CK;

  // ---- every load that needs no other goes out first
  double own[R], ub[R], ra[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW, rr = r < NR ? r : 0;
    own[q] = gld(a.us + (size_t)rr * K, ee);
  }
  // the neighbours' slots of this thread's rows, and its own point's side
  int nbq[RN];
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW, rr = r < 3 * NR ? r : 0;
    nbq[q] = a.m.slot[(size_t)(rr / NR) * K + ee].x;
  }
  const bool is_side = t < EB * NS, is_vol = !is_side && t < EB * (NS + NQ);
  const int sp = is_side ? row : 0, sk = sp / NQ1, jj = sp - sk * NQ1;
  const int vj = is_vol ? row - NS : 0;
  int2 sl = a.m.slot[(size_t)sk * K + ee];
  const double xr = gld(a.m.xr, ee), yr = gld(a.m.yr, ee);
  const double xs = gld(a.m.xs, ee), ys = gld(a.m.ys, ee);
  double eps_me = 1., eps_nb = 1.;
  if constexpr (PHYS == PH_TE) eps_me = gld(a.m.eps, ee);
  int fl_me = 0;
  if constexpr (has_positivity<PHYS>()) fl_me = gld_int(a.bad, ee);
  double Vv[6] = {0., 0., 0., 0., 0., 0.};
  const bool vary = PHYS == PH_ADV && a.ph.prob == PB_ADV_ROTHILL;
  if (TDB || vary) {
#pragma unroll
    for (int q = 0; q < 6; q++) Vv[q] = gld(a.m.V + (size_t)q * K, ee);
  }
  // the step base and the running combination (used at the end)
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW, rr = r < NR ? r : 0;
    ub[q] = ra[q] = 0.;
    if (use_un || a.conv) ub[q] = gld(a.un + (size_t)rr * K, ee);
    if (a.accmode == ACC_ADD3 || a.accmode == ACC_FINAL6) ra[q] = gld(a.acc + (size_t)rr * K, ee);
  }
  // the step state; the first stage of a step closes the step before it
  DevState S = a.st[(a.step_pos == STEP_MID || a.step_pos == STEP_LAST) ? 1 : 0];
  constexpr int kU = kSmallFold / T;
  unsigned long long pl[kU], pc[kU];
#pragma unroll
  for (int u = 0; u < kU; u++) {
    const int b = t + u * T;
    pl[u] = pc[u] = 0ull;
    if (a.step_pos == STEP_FIRST && b < a.nblk) {
      pl[u] = a.part[b];
      if (a.conv_run) pc[u] = a.part[a.nblk + b];
    }
  }
  for (int q = t; q < NP * NQ; q += T) {
    s_B[q] = TC::B[q];
    s_GX[q] = TC::GX[q];
    s_GY[q] = TC::GY[q];
  }
  for (int q = t; q < 3 * NP * NQ1; q += T) s_side[q] = TC::SIDE[q];

  // ---- the neighbours' coefficients and this point's side
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW;
    if (r < 3 * NR) {
      const int nr = r % NR;
      double v = 0.;
      if (nbq[q] >= 0) {
        v = gld(a.us + (size_t)nr * K, nbq[q]);
        // a flagged neighbour contributes its means only
        if constexpr (has_positivity<PHYS>()) {
          if (a.fix_in && nr % NP != 0 && gld_int(a.bad, nbq[q])) v = 0.;
        }
      }
      s_n[r][el] = v;
    }
  }
  double nx = 0., ny = 0., len = 0., bv[NMAX] = {0., 0., 0., 0.};
  if (is_side) {
    const int sid = sl.y >> 3;
    nx = gld(a.m.snx, sid);
    ny = gld(a.m.sny, sid);
    len = gld(a.m.slen, sid);
    if constexpr (PHYS == PH_TE) eps_nb = sl.x >= 0 ? gld(a.m.eps, sl.x) : eps_me;
    if (sl.x < 0 && !(TDB && sl.x != -1)) {
      const double *b = a.m.bnd_val + ((size_t)a.m.side[sid].w * NQ1 + jj) * NMAX;
#pragma unroll
      for (int n = 0; n < N; n++) bv[n] = b[n];
    }
  }
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW;
    if constexpr (has_positivity<PHYS>()) {
      if (a.fix_in && fl_me && r % NP != 0) own[q] = 0.;
    }
    if (r < NR) s_c[r][el] = own[q];
  }
  if (a.step_pos == STEP_FIRST) {
    unsigned long long kl = pl[0], kc = pc[0];
#pragma unroll
    for (int u = 1; u < kU; u++) {
      kl = pl[u] > kl ? pl[u] : kl;
      kc = pc[u] > kc ? pc[u] : kc;
    }
    kl = wave_max_key(kl);
    kc = wave_max_key(kc);
    if ((t & 63) == 0) {
      s_l[t >> 6] = kl;
      s_k[t >> 6] = kc;
    }
  }
  __syncthreads();
  if (a.step_pos == STEP_FIRST) {
    if (S.pending && !(S.nan_flag | S.halt)) {
      unsigned long long kl = s_l[0], kc = s_k[0];
#pragma unroll
      for (int w = 1; w < T / 64; w++) {
        kl = s_l[w] > kl ? s_l[w] : kl;
        kc = s_k[w] > kc ? s_k[w] : kc;
      }
      S.pending = 0;
      FinishArgs f;
      f.cfl_mode = a.cfl_mode;
      f.cfl_num = a.cfl_num;
      f.p = P;
      f.fixed_dt = 0.;
      f.initial = 0;
      f.t0 = 0.;
      f.conv = a.conv_run;
      close_step(S, ord_val(kl), ord_val(kc), f, 0.);
    }
    if (blockIdx.x == 0 && t == 0) a.st[1] = S;
  }
  if (a.step_pos == STEP_LAST && blockIdx.x == 0 && t == 0) {
    DevState B = S;
    B.pending = !(S.nan_flag | S.halt);
    a.st[0] = B;
  }
  if (S.nan_flag | S.halt) return;
  const double dt = S.dt;

  // ---- points
  if (is_side) {
    // eval_surface conserv_kernels.cu:850-985 at point jj of local side sk;
    // the neighbour walks the side the other way
    const int nb = sl.x, nbls = sl.y & 3, role = (sl.y >> 2) & 1;
    double Um[NMAX], Un[NMAX], F[NMAX];
    const double *po = s_side + (size_t)(sk * NP) * NQ1 + jj;
    const double *pn = s_side + (size_t)(nbls * NP) * NQ1 + NQ1 - 1 - jj;
#pragma unroll
    for (int n = 0; n < N; n++) {
      Um[n] = s_c[n * NP][el] * po[0];
      Un[n] = s_n[sk * NR + n * NP][el] * pn[0];
    }
#pragma unroll
    for (int i = 1; i < NP; i++) {
      const double x = po[i * NQ1], y = pn[i * NQ1];
#pragma unroll
      for (int n = 0; n < N; n++) {
        Um[n] = fma(s_c[n * NP + i][el], x, Um[n]);
        Un[n] = fma(s_n[sk * NR + n * NP + i][el], y, Un[n]);
      }
    }
    if (nb < 0) {
      if (nb == -1) {
        wall_state<PHYS>(a.ph, Um, Un, bv[0], bv[1], bv[2]);
      } else {
        if constexpr (TDB) {
          double x, y;
          side_point<NQ1>(Vv, TC::X1, sk, jj, x, y);
          boundary_data<PHYS>(a.ph, x, y, S.t + a.cstage * dt, nx, ny, -nb, bv);
        }
#pragma unroll
        for (int n = 0; n < N; n++) Un[n] = bv[n];
      }
    }
    double f;
    const double w1 = TC::W1[jj];
    if constexpr (llf_only<PHYS>()) {
      riemann<PHYS>(a.ph, Um, Un, role ? -nx : nx, role ? -ny : ny, 1., 1., F);
      f = -0.5 * len * w1;
    } else {
      double UL[NMAX], UR[NMAX];
#pragma unroll
      for (int n = 0; n < N; n++) {
        UL[n] = role ? Un[n] : Um[n];
        UR[n] = role ? Um[n] : Un[n];
      }
      PhysParams pv = a.ph;
      if constexpr (PHYS == PH_ADV) {
        if (vary) {
          double x, y;
          side_point<NQ1>(Vv, TC::X1, sk, jj, x, y);
          rothill_velocity(x, y, pv.ax, pv.ay);
        }
      }
      riemann<PHYS>(pv, UL, UR, nx, ny, role ? eps_nb : eps_me, role ? eps_me : eps_nb, F);
      f = (role ? 0.5 : -0.5) * len * w1;
    }
#pragma unroll
    for (int n = 0; n < N; n++) s_f[sp][n][el] = F[n] * f;
  } else if (is_vol) {
    // eval_volume conserv_kernels.cu:1042-1081 at point vj
    double U[NMAX], ga[NMAX], gb[NMAX];
#pragma unroll
    for (int n = 0; n < N; n++) U[n] = s_c[n * NP][el] * s_B[vj];
#pragma unroll
    for (int i = 1; i < NP; i++) {
      const double x = s_B[i * NQ + vj];
#pragma unroll
      for (int n = 0; n < N; n++) U[n] = fma(s_c[n * NP + i][el], x, U[n]);
    }
    PhysParams pv = a.ph;
    if constexpr (PHYS == PH_ADV) {
      if (vary) {
        double x, y;
        elem_point(Vv, TC::R1[vj], TC::R2[vj], x, y);
        rothill_velocity(x, y, pv.ax, pv.ay);
      }
    }
    flux_contra<PHYS>(pv, U, xr, yr, xs, ys, ga, gb);
#pragma unroll
    for (int n = 0; n < N; n++) {
      s_g[vj][0][n][el] = ga[n];
      s_g[vj][1][n][el] = gb[n];
    }
  }
  __syncthreads();

  // ---- modes: k = dt/J (surface + volume), then the RK combination
  const double sdt = dt / __dsub_rn(__dmul_rn(xr, ys), __dmul_rn(xs, yr));
  double o[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW, n = r < NR ? r / NP : 0, i = r < NR ? r % NP : 0;
    double acc = 0.;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int j = 0; j < NQ1; j++)
        acc = fma(s_f[k * NQ1 + j][n][el], s_side[(k * NP + i) * NQ1 + j], acc);
#pragma unroll
    for (int j = 0; j < NQ; j++)
      acc = fma(s_GX[i * NQ + j], s_g[j][0][n][el], fma(s_GY[i * NQ + j], s_g[j][1][n][el], acc));
    double sc = sdt;
    if constexpr (PHYS == PH_TE) sc = sdt * (n < 2 ? 1. / eps_me : 1. / a.ph.mu);
    acc *= sc;
    const bool mine = act && r < NR;
    if constexpr (PHYS == PH_TE) {
      if (a.kout && mine && n < 2) gst(a.kout + (size_t)r * K, e, acc);
    }
    const double us = own[q];
    double un = ub[q];
    if constexpr (has_positivity<PHYS>()) {
      if (a.fix_un && fl_me && i != 0) un = 0.;
    }
    if (a.accmode == ACC_FINAL6) {
      o[q] = un + (ra[q] + acc * (1. / 6.));
    } else {
      if (a.accmode == ACC_SET6 && mine) gst(a.acc + (size_t)r * K, e, acc * (1. / 6.));
      if (a.accmode == ACC_ADD3 && mine) gst(a.acc + (size_t)r * K, e, ra[q] + acc * (1. / 3.));
      if (a.mode == M_US_CK)
        o[q] = us + a.C * acc;
      else if (a.mode == M_A_UN_B_US_CK)
        o[q] = (a.A * un + a.B * us) + a.C * acc;
      else if (a.mode == M_UN_CK)
        o[q] = un + a.C * acc;
      else
        o[q] = acc;
    }
  }
  // the new coefficients together, where the element as a whole is asked for:
  // the positivity check of what is stored, the CFL speed
  const bool check = has_positivity<PHYS>() && (a.fix_out || (a.last_stage && a.flags_out));
  if (check || a.last_stage) {
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int r = row + q * RW;
      if (r < NR) s_c[r][el] = o[q];  // (read last before the barrier above)
    }
    __syncthreads();
  }
  if constexpr (has_positivity<PHYS>()) {
    if (check) {
      const bool bad = small_needs_fix<PHYS, P, EB>(a.ph, s_c, s_B, s_side, s_md, s_bad, el, row);
      if (a.fix_out && bad) {
#pragma unroll
        for (int q = 0; q < R; q++)
          if ((row + q * RW) % NP != 0) o[q] = 0.;
      }
      if (row == 0 && act) {
        if (a.last_stage && a.flags_out) a.bad[e] = bad ? 1 : 0;
        if (bad && a.fired) atomicOr(a.fired, 1);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW;
    if (act && r < NR) gst(a.out + (size_t)r * K, e, o[q]);
  }
  if (a.last_stage) {
    // step-to-step change over rows r < N (time_integrator.cu:404-414)
    if (a.conv) {
      double dc = 0.;
#pragma unroll
      for (int q = 0; q < R; q++)
        if (act && row + q * RW < (N < NR ? N : NR)) dc = fmax(dc, fabs(o[q] - ub[q]));
      const unsigned long long kc = wave_max_key(ord_key(dc));
      if ((t & 63) == 0) s_k[t >> 6] = kc;
      __syncthreads();
    }
    double lam = 0.;
    if (a.cfl_mode && act && row == 0) {
      double U[NMAX];
#pragma unroll
      for (int n = 0; n < N; n++) U[n] = s_c[n * NP][el] * TC::B[0];
      PhysParams pv = a.ph;
      if constexpr (PHYS == PH_ADV) {
        if (vary) {
          double x, y;
          elem_point(Vv, TC::R1[NQ / 2], TC::R2[NQ / 2], x, y);
          rothill_velocity(x, y, pv.ax, pv.ay);
        }
      }
      lam = ref_max_operand(cfl_speed<PHYS>(pv, U, eps_me), e);
    }
    if (t < 64) {  // row 0 lies in the first wave
      const unsigned long long kl = wave_max_key(ord_key(lam));
      if (t == 0) {
        a.part[blockIdx.x] = kl;
        if (a.conv) {
          unsigned long long kc = s_k[0];
#pragma unroll
          for (int w = 1; w < T / 64; w++) kc = s_k[w] > kc ? s_k[w] : kc;
          a.part[a.nblk + blockIdx.x] = kc;
        }
      }
    }
  }
}

}  // namespace dgk

// dg_stage_s.h -- the RK stage on small meshes: a thread per point, then a
// thread per coefficient.
//
// On a mesh of a few thousand elements the one-thread-per-element stage is a
// single wave on a few CUs that walks tens of kilobytes of straight-line code
// (every table entry an immediate), so its time is the instruction stream of
// one wave and the chip idles.  Here a block takes EB elements:
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
// partials, block 0 stores the new step state), and for advection and Euler
// time-dependent boundary data are evaluated by the side points that use them.
// Bound by latency: of 8.4 us per stage (supersonic vortex p = 3 on 2,880
// triangles; 22.9 on the one-thread kernel with its boundary and close) 2.4 are
// the launch, 2.6 the two dependent memory round trips and the store, the rest
// the points, the modes and the positivity check.  Rotating hill p = 4 on 1,080
// triangles: 26.4 -> 6.2 us.  (Fewer elements per block fill more CUs, but
// below the widths here the loads fall under 32 B per row.)
#pragma once

#include "dg_stage.h"

namespace dgk {

// elements per block, and its threads: a thread per point, the side points in
// whole waves of their own (a wave with both would run one's code after the
// other's), and a thread per coefficient (a second pass over them for the last
// few doubles the modes' latency).  us per SSP-RK3 stage, Euler: p = 3 with 320
// threads for its 320 coefficients 8.8 on 2,888 triangles, with 256 9.6.  At
// p = 4 the second pass is nearly full and 256 threads are better than 512
// (6,050 triangles 14.6 / 17.2).  At p = 2 the separate waves and the single
// pass (384 threads, FULL) are better while the chip has room for them (2,888:
// 7.2, with 256 7.9) and worse once it is full (16,200: 15.4 / 13.5): FULL is
// for up to two blocks per CU.  The VJP at Euler p = 5 keeps the second pass
// too: its flux adjoint spills in the registers that 384 threads leave (3,872:
// 104.9 us a reverse stage; 66.9).
__host__ __device__ constexpr int small_eb(int p) {
  return p == 0 ? 64 : p <= 2 ? 16 : p <= 4 ? 8 : 4;
}
template <int P, bool FULL>
__host__ __device__ constexpr int small_side_t() {  // threads before the volume points
  constexpr int n = small_eb(P) * 3 * (P + 1);
  return FULL ? (n + 63) / 64 * 64 : n;
}
template <int PHYS, int P, bool FULL, bool VJP = false>
__host__ __device__ constexpr int small_t() {
  constexpr int eb = small_eb(P), pts = small_side_t<P, FULL>() + eb * nq_of(P);
  constexpr int rows = FULL && P != 4 && !(VJP && P == 5) ? eb * nvars_of(PHYS) * np_of(P) : 0;
  return ((pts > rows ? pts : rows) + 63) / 64 * 64;
}
__host__ __device__ constexpr bool small_full(int p, int nblk) { return p != 2 || nblk <= 512; }

// An element's variables lie together in LDS, in pairs that one 16-byte access
// moves (three variables are padded to four): b64 accesses were most of the
// points' time.
template <int PHYS>
__host__ __device__ constexpr int small_nv() {
  return nvars_of(PHYS) == 1 ? 1 : 4;
}
template <int N, int NV>
__device__ __forceinline__ void lds_get(const double (&s)[NV], double *v) {
  if constexpr (NV == 1) {
    v[0] = s[0];
  } else {
    const dbl2 a = *(const dbl2 *)&s[0], b = *(const dbl2 *)&s[2];
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    if constexpr (N == 4) v[3] = b.y;
  }
}
template <int N, int NV>
__device__ __forceinline__ void lds_put(double (&s)[NV], const double *v) {
  if constexpr (NV == 1) {
    s[0] = v[0];
  } else {
    *(dbl2 *)&s[0] = dbl2{v[0], v[1]};
    *(dbl2 *)&s[2] = dbl2{v[2], N == 4 ? v[3] : 0.};
  }
}

// needs_fix of the block's elements' new coefficients s_c (element-local
// positivity): rows 0 .. N-1 bound one variable each and every thread of an
// element takes the same decision from the bounds; where they do not settle
// it (rare), each thread checks one of its element's points
template <int PHYS, int P, int EB>
__device__ __forceinline__ bool small_needs_fix(const PhysParams &ph,
                                                const double (*s_c)[EB][small_nv<PHYS>()],
                                                const double *s_B, const double *s_side,
                                                double (*s_md)[nvars_of(PHYS)][EB], int *s_bad,
                                                int el, int row) {
  using TC = TabC<P>;
  constexpr int NP = TC::NP, NQ = TC::NQ, NQ1 = TC::NQ1, N = nvars_of(PHYS);
  constexpr double margin = 1e-10;
  if (row < N) {
    double d = 0.;
#pragma unroll
    for (int i = 1; i < NP; i++) d = fma(fabs(s_c[i][el][row]), phi_bound<P>(i), d);
    s_md[0][row][el] = s_c[0][el][row] * TC::B[0];
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
      for (int n = 0; n < N; n++) U[n] = fma(s_c[i][el][n], t[i * st], U[n]);
    if (!is_physical<PHYS>(ph, U)) s_bad[el] = 1;  // (every writer stores the same value)
  }
  __syncthreads();
  return s_bad[el] != 0;
}

// the systems whose stage has the TDB form (outside states that depend on
// time, evaluated by the side points): those that the moving problems are
// states of.  The others run a moving problem too, with a launch before the
// stage (launch_stage_bnd).
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
template <int PHYS, int P, bool TDB, bool FULL>
__global__ __launch_bounds__((small_t<PHYS, P, FULL>())) void k_stage_s(const StageArgs a) {
  using TC = TabC<P>;
  constexpr int NP = TC::NP, NQ = TC::NQ, NQ1 = TC::NQ1, N = nvars_of(PHYS);
  constexpr int EB = small_eb(P), NR = N * NP, NS = 3 * NQ1, T = small_t<PHYS, P, FULL>();
  constexpr int RW = T / EB;                 // rows of one pass over the elements
  constexpr int R = (NR + RW - 1) / RW;      // passes over the own rows
  constexpr int RN = (3 * NR + RW - 1) / RW;  // and over the neighbours'
  constexpr int SV = small_side_t<P, FULL>();  // the first volume point's thread
  static_assert(SV + EB * NQ <= T && SV % EB == 0 && NQ + NS <= RW, "a thread per point");
  constexpr int NV = small_nv<PHYS>();
  __shared__ double s_B[NP * NQ], s_side[3 * NP * NQ1];
  __shared__ dbl2 s_G[NP * NQ], s_g[NQ][N][EB];  // (r, s) components
  __shared__ __align__(16) double s_c[NP][EB][NV], s_n[3][NP][EB][NV], s_f[NS][EB][NV];
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
  const bool is_side = t < EB * NS, is_vol = t >= SV && t < SV + EB * NQ;
  const int sp = is_side ? row : 0, sk = sp / NQ1, jj = sp - sk * NQ1;
  const int vj = is_vol ? row - SV / EB : 0;
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
  constexpr int kU = (kSmallFold + T - 1) / T;
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
    s_G[q] = dbl2{TC::GX[q], TC::GY[q]};
  }
  for (int q = t; q < 3 * NP * NQ1; q += T) s_side[q] = TC::SIDE[q];

  // ---- the neighbours' coefficients and this point's side, requested
  // together: no branch lies between the loads (a row past the last, a
  // boundary's missing neighbour have stand-ins), as
  // each would make its load a round trip of its own
  const int sid = sl.y >> 3;
  double nbv[RN];
  int fl_nb[RN];
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW, nr = r < 3 * NR ? r % NR : 0;
    const int nb = nbq[q] >= 0 ? nbq[q] : ee;
    nbv[q] = gld(a.us + (size_t)nr * K, nb);
    fl_nb[q] = 0;
  }
  if constexpr (has_positivity<PHYS>()) {
    if (a.fix_in) {
#pragma unroll
      for (int q = 0; q < RN; q++) fl_nb[q] = gld_int(a.bad, nbq[q] >= 0 ? nbq[q] : ee);
    }
  }
  double nx = 0., ny = 0., len = 0., bv[NMAX] = {0., 0., 0., 0.};
  if (is_side) {
    nx = gld(a.m.snx, sid);
    ny = gld(a.m.sny, sid);
    len = gld(a.m.slen, sid);
    const int bslot = a.m.side[sid].w;
    if constexpr (PHYS == PH_TE) eps_nb = gld(a.m.eps, sl.x >= 0 ? sl.x : ee);
    if (sl.x < 0 && !(TDB && sl.x != -1)) {
      const double *b = a.m.bnd_val + ((size_t)bslot * NQ1 + jj) * NMAX;
#pragma unroll
      for (int n = 0; n < N; n++) bv[n] = b[n];
    }
  }
#pragma unroll
  for (int q = 0; q < RN; q++) {
    const int r = row + q * RW, nr = r % NR;
    // a flagged neighbour contributes its means only
    const bool zero = nbq[q] < 0 || (fl_nb[q] && nr % NP != 0);
    if (r < 3 * NR) s_n[r / NR][nr % NP][el][nr / NP] = zero ? 0. : nbv[q];
  }
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = row + q * RW;
    if constexpr (has_positivity<PHYS>()) {
      if (a.fix_in && fl_me && r % NP != 0) own[q] = 0.;
    }
    if (r < NR) s_c[r % NP][el][r / NP] = own[q];
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
    for (int i = 0; i < NP; i++) {
      const double x = po[i * NQ1], y = pn[i * NQ1];
      double cm[N], cn[N];
      lds_get<N>(s_c[i][el], cm);
      lds_get<N>(s_n[sk][i][el], cn);
#pragma unroll
      for (int n = 0; n < N; n++) {
        Um[n] = i ? fma(cm[n], x, Um[n]) : cm[n] * x;
        Un[n] = i ? fma(cn[n], y, Un[n]) : cn[n] * y;
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
    for (int n = 0; n < N; n++) F[n] *= f;
    lds_put<N>(s_f[sp][el], F);
  } else if (is_vol) {
    // eval_volume conserv_kernels.cu:1042-1081 at point vj
    double U[NMAX], ga[NMAX], gb[NMAX];
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const double x = s_B[i * NQ + vj];
      double cm[N];
      lds_get<N>(s_c[i][el], cm);
#pragma unroll
      for (int n = 0; n < N; n++) U[n] = i ? fma(cm[n], x, U[n]) : cm[n] * x;
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
    for (int n = 0; n < N; n++) s_g[vj][n][el] = dbl2{ga[n], gb[n]};
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
        acc = fma(s_f[k * NQ1 + j][el][n], s_side[(k * NP + i) * NQ1 + j], acc);
#pragma unroll
    for (int j = 0; j < NQ; j++) {
      const dbl2 G = s_G[i * NQ + j], g = s_g[j][n][el];
      acc = fma(G.x, g.x, fma(G.y, g.y, acc));
    }
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
      if (r < NR) s_c[r % NP][el][r / NP] = o[q];  // (read last before the barrier above)
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
      for (int n = 0; n < N; n++) U[n] = s_c[0][el][n] * TC::B[0];
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

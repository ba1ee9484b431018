// Structured linear algebra and the Rodas5 step for one wave-resident mode.
//
// W = I/(gamma h) - J with J split as
//   J = [ g'(a)    0   0    ]   rows/cols: a (slot 0 lane 0),
//       [ J_1a     0   c_1^T]              a*h' accumulator (lane 1),
//       [ J_Ra     0   B + U C^T ]         the rest (R)
// B is block-tridiagonal along the lane chains (plus the delta_gamma leaf),
// U C^T is the rank-3 coupling through h', eta' and Pi.  Solve: k_a first
// (scalar), then W_B^{-1} by parallel cyclic reduction with a Woodbury
// correction, then k_1 (a*h' is never read by any other row).
#pragma once

#include "deb_mode.h"

namespace deb {

// wave-uniform step factors of Mode
struct ModeU {
  double gh;         // gamma * h
  double inv_kaden;  // 1 / (1/(gamma h) - g')
  double J1a;
  double leafm, wdg, ddg;  // leaf elimination: W_tg,dg / d_dg, W_dg,tg, 1/d_dg
  double Sinv[3][3];
  double c1Z[3];
};
typedef DEB_LDS ModeU lds_mode_u;

template <int NS>
struct Mode {
  uint32_t rd[NS];
  RowK<NS> rk;       // the rows' constants (row_consts)
  BgCache bg;        // the background's constants and spline windows (bg_init)
  // PCR factors of W_B: d' = sig*d + al*d[i-s] + be*d[i+s] at level s = 2^L;
  // al and be live in the wave's LDS ([PCR_LEVELS][2][NS][64], pcr_lds_doubles)
  lds_double *pcr;
  __device__ __forceinline__ lds_double &al(int L, int j) const { return pcr[((L * 2) * NS + j) * WAVE + lane_id()]; }
  __device__ __forceinline__ lds_double &be(int L, int j) const {
    return pcr[((L * 2 + 1) * NS + j) * WAVE + lane_id()];
  }
  double sig0[NS];
  double binv[NS];
  double Z[3][NS];   // W_B^{-1} [u_h, u_eta, u_pi]
  double Cf[3][NS];  // c_h, c_eta, c_pi
  double c1[NS];
  double U[3][NS];   // u_h, u_eta, u_pi (where h', eta', Pi enter each row)
  double jcol[NS];   // df/da at the step start
  // the wave-uniform factors, in the wave's LDS (one copy per wave rather than
  // one per lane in registers or scratch)
  lds_mode_u *u;
  int nlev;
};

// evaluate f (T-valued) at (tau, y) and the coefficient rows cf
template <int NS, typename T>
__device__ __forceinline__ void eval_rhs(BgCache &bg, const RowK<NS> &K, double tau, const double (&y)[NS],
                                         T (&f)[NS], Coef<T> (&cf)[NS]) {
  const int lane = lane_id();
  double a0 = readlane(y[0], L_A);
  T a;
  if constexpr (sizeof(T) == sizeof(double)) a = a0; else a = T{a0, 1.0};
  const BgRow<T> b = background_row(bg, a);
  const double invtau = rcp_nr(tau);
#pragma unroll
  for (int s = 0; s < NS; ++s) cf[s] = row_lin<NS, T>(K, s, b, bg, invtau);
  // functionals h', eta', Pi, f_1
  constexpr int NV = (sizeof(T) == sizeof(double)) ? 4 : 8;
  double part[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) part[i] = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    part[0] += vval(cf[s].ch) * y[s];
    part[1] += vval(cf[s].ceta) * y[s];
    part[2] += vval(cf[s].cpi) * y[s];
    part[3] += vval(cf[s].c1) * y[s];
    if constexpr (NV == 8) {
      part[4] += dval(cf[s].ch) * y[s];
      part[5] += dval(cf[s].ceta) * y[s];
      part[6] += dval(cf[s].cpi) * y[s];
      part[7] += dval(cf[s].c1) * y[s];
    }
  }
  if constexpr (NV == 4) wave_sum4(part);
  else wave_sum<NV>(part);
  T hp, etap, Pi, f1;
  if constexpr (NV == 8) {
    hp = T{part[0], part[4]};
    etap = T{part[1], part[5]};
    Pi = T{part[2], part[6]};
    f1 = T{part[3], part[7]};
  } else {
    hp = part[0];
    etap = part[1];
    Pi = part[2];
    f1 = part[3];
  }
  const double ydg = readlane(y[0], L_DG), ytg = readlane(y[0], L_TG);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    double ym = from_prev(y[s]);
    double yp = from_next(y[s]);
    const Coef<T> &r = cf[s];
    T v = r.sub * ym + r.diag * y[s] + r.sup * yp + r.uh * hp + r.ueta * etap + r.upi * Pi;
    if (s == 0) {
      if (lane == L_DG) v = v + r.leaf * ytg;
      if (lane == L_TG) v = v + r.leaf * ydg;
      if (lane == L_A) v = b.aH * b.a;
      if (lane == L_AHP) v = f1;
    }
    f[s] = v;
  }
}
template <int NS>
__device__ __forceinline__ void eval_rhs(BgCache &bg, const RowK<NS> &K, double tau, const double (&y)[NS],
                                         double (&f)[NS]) {
  Coef<double> cf[NS];
  eval_rhs<NS, double>(bg, K, tau, y, f, cf);
}

// df/dtau: only the hierarchy truncation rows depend on tau explicitly
template <int NS>
__device__ __forceinline__ void dfdtau(const RowK<NS> &K, double tau, const double (&y)[NS], double (&dT)[NS]) {
  const double it = 1.0 / tau, it2 = it * it;
#pragma unroll
  for (int s = 0; s < NS; ++s) dT[s] = K.tr[s] != 0.0 ? K.tr[s] * it2 * y[s] : 0.0;
}

// W_B^{-1} r (leaf elimination + PCR)
template <int NS>
__device__ __forceinline__ void bsolve(const Mode<NS> &m, double (&x)[NS]) {
  const int lane = lane_id();
  const double rdg = readlane(x[0], L_DG);
  if (lane == L_TG) x[0] -= m.u->leafm * rdg;
#pragma unroll
  for (int L = 0; L < PCR_LEVELS; ++L) {
    if (L >= m.nlev) break;
    const int s = 1 << L;
    if (L == PCR_LAST) {
#pragma unroll
      for (int j = 0; j < NS; ++j) x[j] += m.al(L, j) * from_lane(x[j], lane ^ 32);
      break;
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      double dm, dp;
      if (L == 0) {
        dm = from_prev(x[j]);
        dp = from_next(x[j]);
      } else {
        int lm = lane - s < 0 ? 0 : lane - s;
        int lp = lane + s > WAVE - 1 ? WAVE - 1 : lane + s;
        dm = from_lane(x[j], lm);
        dp = from_lane(x[j], lp);
      }
      double sg = (L == 0) ? m.sig0[j] : 1.0;
      x[j] = sg * x[j] + m.al(L, j) * dm + m.be(L, j) * dp;
    }
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) x[j] *= m.binv[j];
  const double xtg = readlane(x[0], L_TG);
  if (lane == L_DG) x[0] = (rdg - m.u->wdg * xtg) * m.u->ddg;
}

// factorisation of W at (tau0, y0) for step size h; f0 = f(tau0, y0)
template <int NS>
__device__ __forceinline__ void factor(Mode<NS> &m, double tau0, const double (&y0)[NS], double h,
                                       double (&f0)[NS]) {
  const int lane = lane_id();
  constexpr double gamma = 0.19;
  dual fd[NS];
  Coef<dual> co[NS];
  eval_rhs<NS, dual>(m.bg, m.rk, tau0, y0, fd, co);
#pragma unroll
  for (int s = 0; s < NS; ++s) f0[s] = fd[s].v;
  m.u->gh = gamma * h;
  const double igh = 1.0 / m.u->gh;
  double gprime = readlane(fd[0].d, L_A);
  m.u->J1a = readlane(fd[0].d, L_AHP);
  m.u->inv_kaden = 1.0 / (igh - gprime);
  double A[NS], Bd[NS], Cc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    // the a-row and the a*h' row are solved apart (unused lanes hold zero rows)
    const bool special = s == 0 && lane <= L_AHP;
    m.jcol[s] = special ? 0.0 : fd[s].d;
    A[s] = special ? 0.0 : -co[s].sub.v;
    Cc[s] = special ? 0.0 : -co[s].sup.v;
    Bd[s] = special ? 1.0 : igh - co[s].diag.v;
    m.Cf[0][s] = co[s].ch.v;
    m.Cf[1][s] = co[s].ceta.v;
    m.Cf[2][s] = co[s].cpi.v;
    m.c1[s] = co[s].c1.v;
    m.U[0][s] = co[s].uh.v;
    m.U[1][s] = co[s].ueta.v;
    m.U[2][s] = co[s].upi.v;
  }
  // leaf: delta_gamma (lane L_DG) couples only to theta_gamma (lane L_TG)
  const double w_dg_tg = -readlane(co[0].leaf.v, L_DG);
  const double w_tg_dg = -readlane(co[0].leaf.v, L_TG);
  m.u->ddg = m.u->gh;  // 1 / d_dg with d_dg = 1/(gamma h)
  m.u->wdg = w_dg_tg;
  m.u->leafm = w_tg_dg * m.u->gh;
  if (lane == L_TG) Bd[0] -= w_tg_dg * w_dg_tg * m.u->gh;
  // PCR factorisation; the dark-energy 2x2 block (lanes L_DQ, L_TQ of slot 0)
  // is eliminated at level 0 by cross-multiplication (its theta_Q pivot can
  // vanish), every other row by the usual reduction, which multiplies by the
  // neighbours' pivot reciprocals (each lane takes the reciprocal of its own
  // pivot once per level).  A row that is not coupled to a neighbour has a zero
  // coefficient, so its products vanish; only the dark-energy pivots of slot 0
  // can be infinite there, and those are guarded at level 0.
#pragma unroll
  for (int L = 0; L < PCR_LEVELS; ++L) {
    if (L >= m.nlev) break;
    const int s = 1 << L;
    if (L == PCR_LAST) {
      // lanes below 32 have only the neighbour above, the others only the one below
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const double E = lane < 32 ? Cc[j] : A[j];
        const double al = -E * from_lane(rcp_nr(Bd[j]), lane ^ 32);
        m.al(L, j) = al;
        Bd[j] += al * from_lane(E, lane ^ 32);
      }
      break;
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const double ib = rcp_nr(Bd[j]);
      double am, ibm, cm, ap, ibp, cp;
      if (L == 0) {
        am = from_prev(A[j]); ibm = from_prev(ib); cm = from_prev(Cc[j]);
        ap = from_next(A[j]); ibp = from_next(ib); cp = from_next(Cc[j]);
      } else {
        int lm = lane - s < 0 ? 0 : lane - s;
        int lp = lane + s > WAVE - 1 ? WAVE - 1 : lane + s;
        am = from_lane(A[j], lm); ibm = from_lane(ib, lm); cm = from_lane(Cc[j], lm);
        ap = from_lane(A[j], lp); ibp = from_lane(ib, lp); cp = from_lane(Cc[j], lp);
      }
      double alpha = -A[j] * ibm, beta = -Cc[j] * ibp;
      if (L == 0 && j == 0) {
        alpha = A[j] == 0.0 ? 0.0 : alpha;
        beta = Cc[j] == 0.0 ? 0.0 : beta;
      }
      double sg = 1.0;
      if (L == 0 && j == 0) {
        // scale the row by the partner's pivot instead of dividing by it
        const double bm = from_prev(Bd[0]), bp = from_next(Bd[0]);
        if (lane == L_DQ) { sg = bp; beta = -Cc[j]; alpha = 0.0; }
        if (lane == L_TQ) { sg = bm; alpha = -A[j]; beta = 0.0; }
      }
      double nb = sg * Bd[j] + alpha * cm + beta * ap;
      double na = alpha * am;
      double nc = beta * cp;
      m.al(L, j) = alpha;
      m.be(L, j) = beta;
      if (L == 0) m.sig0[j] = sg;
      Bd[j] = nb;
      A[j] = na;
      Cc[j] = nc;
    }
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) m.binv[j] = rcp_nr(Bd[j]);
  // Woodbury: Z = W_B^{-1} U, S = I - C^T Z
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    double x[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const bool special = s == 0 && lane <= L_AHP;
      double u = r == 0 ? co[s].uh.v : (r == 1 ? co[s].ueta.v : co[s].upi.v);
      x[s] = special ? 0.0 : u;
    }
    bsolve<NS>(m, x);
#pragma unroll
    for (int s = 0; s < NS; ++s) m.Z[r][s] = x[s];
  }
  double part[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) part[i] = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
#pragma unroll
      for (int c = 0; c < 3; ++c) part[r * 3 + c] += m.Cf[r][s] * m.Z[c][s];
      part[9 + r] += m.c1[s] * m.Z[r][s];
    }
  }
  {
    const double t = wave_sum_spread(part);
#pragma unroll
    for (int i = 0; i < 12; ++i) part[i] = readlane(t, i);
  }
  double S[3][3];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) S[r][c] = (r == c ? 1.0 : 0.0) - part[r * 3 + c];
  const double det = S[0][0] * (S[1][1] * S[2][2] - S[1][2] * S[2][1]) -
                     S[0][1] * (S[1][0] * S[2][2] - S[1][2] * S[2][0]) +
                     S[0][2] * (S[1][0] * S[2][1] - S[1][1] * S[2][0]);
  const double id = 1.0 / det;
  m.u->Sinv[0][0] = (S[1][1] * S[2][2] - S[1][2] * S[2][1]) * id;
  m.u->Sinv[0][1] = (S[0][2] * S[2][1] - S[0][1] * S[2][2]) * id;
  m.u->Sinv[0][2] = (S[0][1] * S[1][2] - S[0][2] * S[1][1]) * id;
  m.u->Sinv[1][0] = (S[1][2] * S[2][0] - S[1][0] * S[2][2]) * id;
  m.u->Sinv[1][1] = (S[0][0] * S[2][2] - S[0][2] * S[2][0]) * id;
  m.u->Sinv[1][2] = (S[0][2] * S[1][0] - S[0][0] * S[1][2]) * id;
  m.u->Sinv[2][0] = (S[1][0] * S[2][1] - S[1][1] * S[2][0]) * id;
  m.u->Sinv[2][1] = (S[0][1] * S[2][0] - S[0][0] * S[2][1]) * id;
  m.u->Sinv[2][2] = (S[0][0] * S[1][1] - S[0][1] * S[1][0]) * id;
  m.u->c1Z[0] = part[9];
  m.u->c1Z[1] = part[10];
  m.u->c1Z[2] = part[11];
}

// k = W^{-1} r (r is overwritten by k)
template <int NS>
__device__ __forceinline__ void wsolve(const Mode<NS> &m, double (&r)[NS]) {
  const int lane = lane_id();
  const double ra = readlane(r[0], L_A);
  const double r1 = readlane(r[0], L_AHP);
  const double ka = ra * m.u->inv_kaden;
#pragma unroll
  for (int s = 0; s < NS; ++s) r[s] += m.jcol[s] * ka;
  if (lane == L_A || lane == L_AHP) r[0] = 0.0;
  bsolve<NS>(m, r);
  double g[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    g[0] += m.Cf[0][s] * r[s];
    g[1] += m.Cf[1][s] * r[s];
    g[2] += m.Cf[2][s] * r[s];
    g[3] += m.c1[s] * r[s];
  }
  wave_sum4(g);
  double t[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) t[i] = m.u->Sinv[i][0] * g[0] + m.u->Sinv[i][1] * g[1] + m.u->Sinv[i][2] * g[2];
#pragma unroll
  for (int s = 0; s < NS; ++s) r[s] += m.Z[0][s] * t[0] + m.Z[1][s] * t[1] + m.Z[2][s] * t[2];
  const double c1k = g[3] + m.u->c1Z[0] * t[0] + m.u->c1Z[1] * t[1] + m.u->c1Z[2] * t[2];
  const double k1 = m.u->gh * (r1 + m.u->J1a * ka + c1k);
  if (lane == L_A) r[0] = ka;
  if (lane == L_AHP) r[0] = k1;
}

// Rodas5 (W-form) tableau: ode_integrators_stiff.py:622-687
struct R5 {
  static constexpr double gamma = 0.19;
  static constexpr double a21 = 2.0, a31 = 3.040894194418781, a32 = 1.041747909077569, a41 = 2.576417536461461,
                          a42 = 1.622083060776640, a43 = -0.9089668560264532, a51 = 2.760842080225597,
                          a52 = 1.446624659844071, a53 = -0.3036980084553738, a54 = 0.2877498600325443,
                          a61 = -14.09640773051259, a62 = 6.925207756232704, a63 = -41.47510893210728,
                          a64 = 2.343771018586405, a65 = 24.13215229196062;
  static constexpr double C21 = -10.31323885133993, C31 = -21.04823117650003, C32 = -7.234992135176716,
                          C41 = 32.22751541853323, C42 = -4.943732386540191, C43 = 19.44922031041879,
                          C51 = -20.69865579590063, C52 = -8.816374604402768, C53 = 1.260436877740897,
                          C54 = -0.7495647613787146, C61 = -46.22004352711257, C62 = -17.49534862857472,
                          C63 = -289.6389582892057, C64 = 93.60855400400906, C65 = 318.3822534212147,
                          C71 = 34.20013733472935, C72 = -14.15535402717690, C73 = 57.82335640988400,
                          C74 = 25.83362985412365, C75 = 1.408950972071624, C76 = -6.551835421242162,
                          C81 = 42.57076742291101, C82 = -13.80770672017997, C83 = 93.98938432427124,
                          C84 = 18.77919633714503, C85 = -31.58359187223370, C86 = -6.685968952921985,
                          C87 = -5.810979938412932;
  static constexpr double c2 = 0.38, c3 = 0.3878509998321533, c4 = 0.4839718937873840, c5 = 0.4570477008819580;
  static constexpr double d1 = 0.19, d2 = -0.1823079225333714636, d3 = -0.319231832186874912,
                          d4 = 0.3449828624725343, d5 = -0.377417564392089818;
};

// Out-of-line factorisation, for the reverse of a step (next to much other
// live state): as a call, the step factors stay in memory instead of registers.
template <int NS>
__device__ __noinline__ void factor_call(Mode<NS> &m, double tau0, const double (&y0)[NS], double h) {
  double f0[NS];
  factor<NS>(m, tau0, y0, h, f0);
}

// Rodas5 tableau in flattened form (constant memory, read with wave-uniform
// indices): stage point u_i = y0 + sum_j kA[i][j] k_j, y1 = y0 + sum_j kA8[j] k_j,
// stage time t0 + kc[i] h, kd[i] h dT added in stage i, kC[i][j] / h k_j.
__constant__ double kA[8][8] = {
    {0, 0, 0, 0, 0, 0, 0, 0},
    {R5::a21, 0, 0, 0, 0, 0, 0, 0},
    {R5::a31, R5::a32, 0, 0, 0, 0, 0, 0},
    {R5::a41, R5::a42, R5::a43, 0, 0, 0, 0, 0},
    {R5::a51, R5::a52, R5::a53, R5::a54, 0, 0, 0, 0},
    {R5::a61, R5::a62, R5::a63, R5::a64, R5::a65, 0, 0, 0},
    {R5::a61, R5::a62, R5::a63, R5::a64, R5::a65, 1.0, 0, 0},
    {R5::a61, R5::a62, R5::a63, R5::a64, R5::a65, 1.0, 1.0, 0}};
__constant__ double kA8[8] = {R5::a61, R5::a62, R5::a63, R5::a64, R5::a65, 1.0, 1.0, 1.0};
__constant__ double kC[8][8] = {
    {0, 0, 0, 0, 0, 0, 0, 0},
    {R5::C21, 0, 0, 0, 0, 0, 0, 0},
    {R5::C31, R5::C32, 0, 0, 0, 0, 0, 0},
    {R5::C41, R5::C42, R5::C43, 0, 0, 0, 0, 0},
    {R5::C51, R5::C52, R5::C53, R5::C54, 0, 0, 0, 0},
    {R5::C61, R5::C62, R5::C63, R5::C64, R5::C65, 0, 0, 0},
    {R5::C71, R5::C72, R5::C73, R5::C74, R5::C75, R5::C76, 0, 0},
    {R5::C81, R5::C82, R5::C83, R5::C84, R5::C85, R5::C86, R5::C87, 0}};
__constant__ double kc[8] = {0.0, R5::c2, R5::c3, R5::c4, R5::c5, 1.0, 1.0, 1.0};
__constant__ double kd[8] = {R5::d1, R5::d2, R5::d3, R5::d4, R5::d5, 0.0, 0.0, 0.0};

// one Rodas5Transformed step (ode_integrators_stiff.py:718-834): y1 and err = k8;
// st(i, k) sees every stage vector k_{i+1} once it is solved.  The stages run
// as a loop over the tableau: unrolled, the step is about 240 KB of code, four
// times the instruction cache, and every wave fetched it again each step.  A
// single wave's instruction issue bounds it now (64 cosmologies x 256 k at lmax
// 32: 384 ms unrolled, 227 ms as a loop with the rows as constants, 146 ms with
// the register-held background and the split sums).
// Stage 1's right-hand side is the factorisation's.  With kl (the wave's LDS,
// 7 x NS x 64 doubles) the stage vectors k1..k7 are kept there, else in
// registers.
template <int NS, class Store>
__device__ __forceinline__ void rodas5_step_s(Mode<NS> &m, double t0, double dt, const double (&y0)[NS],
                                              double (&y1)[NS], double (&err)[NS], Store st,
                                              lds_double *kl = nullptr) {
  const int lane = lane_id();
  double k[NS], u[NS], f[NS], dT[NS];
  factor<NS>(m, t0, y0, dt, f);
  dfdtau<NS>(m.rk, t0, y0, dT);
  // the stage vectors start from zero: a stage then sums over fixed columns of
  // the tableau (zero from column i on) without meeting what an earlier step,
  // possibly one that was rejected for a non-finite error, left behind
  double kr[7][NS];
#pragma unroll
  for (int j = 0; j < 7; ++j)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (kl) kl[(j * NS + s) * WAVE + lane] = 0.0;
      else kr[j][s] = 0.0;
    }
  auto K = [&](int j, int s) -> double { return kl ? (double)kl[(j * NS + s) * WAVE + lane] : kr[j][s]; };
  const double idt = 1.0 / dt;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    u[s] = y0[s];
    k[s] = 0.0;
  }
#pragma nounroll
  for (int i = 0; i < 8; ++i) {
    double ck[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) ck[s] = 0.0;
    if (i > 0) {
      // u_i, and the sum of the C_ij k_j; from the seventh stage on u_i = u_{i-1} + k_{i-1}
      double du[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) du[s] = i >= 6 ? u[s] + k[s] : y0[s];
      const int ia = i >= 6 ? 0 : i;  // row 0 of the tableau is zero
      auto add = [&](auto first, auto count) {
        constexpr int J0 = decltype(first)::value, NJ = decltype(count)::value;
        double kj[NJ][NS];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int s = 0; s < NS; ++s) kj[j][s] = K(J0 + j, s);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const double aij = kA[ia][J0 + j], cij = kC[i][J0 + j];
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            if (J0 + j < 5) du[s] += aij * kj[j][s];
            ck[s] += cij * kj[j][s];
          }
        }
      };
      add(std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
      if (i > 3) add(std::integral_constant<int, 3>{}, std::integral_constant<int, 4>{});
#pragma unroll
      for (int s = 0; s < NS; ++s) u[s] = du[s];
      eval_rhs<NS>(m.bg, m.rk, t0 + kc[i] * dt, u, f);
    }
    const double hd = dt * kd[i];
#pragma unroll
    for (int s = 0; s < NS; ++s) k[s] = f[s] + hd * dT[s] + idt * ck[s];
    wsolve<NS>(m, k);
    st(i, k);
    if (kl) {
      if (i < 7) {
#pragma unroll
        for (int s = 0; s < NS; ++s) kl[(i * NS + s) * WAVE + lane] = k[s];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (i == j) {
#pragma unroll
          for (int s = 0; s < NS; ++s) kr[j][s] = k[s];
        }
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    err[s] = k[s];
    y1[s] = u[s] + k[s];
  }
}

template <int NS>
__device__ __forceinline__ void rodas5_step(Mode<NS> &m, double t0, double dt, const double (&y0)[NS],
                                            double (&y1)[NS], double (&err)[NS], lds_double *kl = nullptr) {
  rodas5_step_s<NS>(m, t0, dt, y0, y1, err, [](int, const double (&)[NS]) {}, kl);
}

}  // namespace deb

// Reverse-mode (adjoint) building blocks of the gradient path.
//
// The reference differentiates evolve_perturbations with jax.jacfwd
// (nb_minimal_example.ipynb:297) straight through diffrax's loop and
// Rodas5Transformed.step (ode_integrators_stiff.py:718-834).  Here the same
// derivative of the discrete solution is accumulated backwards, one
// wavefront per mode: the accepted states come from the checkpoint tape,
// each step is recomputed and then reversed stage by stage.  The step-size
// controller's decisions carry no derivative; every accepted step keeps its
// fraction of [t0, t1] while t0 (start time), t1 (last output time), the
// initial state, the cosmology scalars and every spline knot move.
//
// Parameter derivatives are projected on up to MAXDIR input tangent
// directions (d cosmo, d tables, d tau_out per direction, supplied by the
// caller): every contraction below runs in dn<1+MAXDIR> arithmetic whose
// component 0 is the derivative along the scale factor a (or tau) and whose
// components 1..MAXDIR are the input tangents.
#pragma once

#include "deb_forward.h"

namespace deb {

constexpr int MAXDIR = DEB_MAXDIR;
using TD = dn<1 + MAXDIR>;          // (a or tau, theta_1..theta_MAXDIR)

// The row passes of the reverse step are real calls rather than inlined:
// inlined into the step they leave one kernel body with thousands of spilled
// registers; as calls each is register-allocated on its own.  An outlined
// function must stay small enough to need no long branches: the compiler's
// long-branch sequences in a non-kernel function were seen to use the return
// address registers s[30:31] without saving them (a wild return).  The
// device-assembly test of the build checks this for every outlined function.
#define DEB_OUTLINE __device__ __noinline__

// ---------------------------------------------------------------------------
// cross-lane moves and reductions of composite scalars, component by
// component (member access only)
template <class T>
struct ncomp;
template <>
struct ncomp<double> { static constexpr int value = 1; };
template <>
struct ncomp<dual> { static constexpr int value = 2; };
template <int N, class B>
struct ncomp<dn<N, B>> { static constexpr int value = (N + 1) * ncomp<B>::value; };

__device__ __forceinline__ double &comp(double &x, int) { return x; }
__device__ __forceinline__ double &comp(dual &x, int i) { return i == 0 ? x.v : x.d; }
template <int N, class B>
__device__ __forceinline__ double &comp(dn<N, B> &x, int i) {
  constexpr int cb = ncomp<B>::value;
  return i < cb ? comp(x.v, i) : comp(x.d[(i - cb) / cb], (i - cb) % cb);
}

template <class T>
__device__ __forceinline__ T t_from_prev(T x) {
#pragma unroll
  for (int i = 0; i < ncomp<T>::value; ++i) comp(x, i) = from_prev(comp(x, i));
  return x;
}
template <class T>
__device__ __forceinline__ T t_from_next(T x) {
#pragma unroll
  for (int i = 0; i < ncomp<T>::value; ++i) comp(x, i) = from_next(comp(x, i));
  return x;
}
template <class T>
__device__ __forceinline__ T t_readlane(T x, int lane) {
#pragma unroll
  for (int i = 0; i < ncomp<T>::value; ++i) comp(x, i) = readlane(comp(x, i), lane);
  return x;
}
// wave-uniform sums of NV composite values
template <class T, int NV>
__device__ __forceinline__ void t_wave_sum(T (&v)[NV]) {
  constexpr int C = ncomp<T>::value;
  double flat[NV * C];
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int i = 0; i < C; ++i) flat[j * C + i] = comp(v[j], i);
  wave_sum<NV * C>(flat);
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int i = 0; i < C; ++i) comp(v[j], i) = flat[j * C + i];
}

// ---------------------------------------------------------------------------
// transposed structured solves: the forward solves' operations in reverse
// order, each replaced by its transpose (same factors, no new factorisation)

// x <- W_B^{-T} x
template <int NS>
__device__ __forceinline__ void bsolveT(const Mode<NS> &m, double (&x)[NS]) {
  const int lane = lane_id();
  // leaf back-substitution x_dg = (r_dg - wdg x_tg) ddg
  const double xdg = readlane(x[0], L_DG);
  double rdgb = m.u->ddg * xdg;
  if (lane == L_TG) x[0] -= m.u->wdg * m.u->ddg * xdg;
  if (lane == L_DG) x[0] = 0.0;
#pragma unroll
  for (int j = 0; j < NS; ++j) x[j] *= m.binv[j];
  // PCR levels in reverse: x_i <- sg_i x_i + al_i x_{i-s} + be_i x_{i+s}
#pragma unroll
  for (int L = PCR_LEVELS - 1; L >= 0; --L) {
    if (L >= m.nlev) continue;
    const int s = 1 << L;
    if (L == PCR_LAST) {
#pragma unroll
      for (int j = 0; j < NS; ++j) x[j] += from_lane(m.al(L, j) * x[j], lane ^ 32);
      continue;
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const double v = m.al(L, j) * x[j];
      const double w = m.be(L, j) * x[j];
      double vn, wp;
      if (L == 0) {
        vn = from_next(v);
        wp = from_prev(w);
      } else {
        const int lp = lane + s, lm = lane - s;
        vn = from_lane(v, lp > WAVE - 1 ? WAVE - 1 : lp);
        wp = from_lane(w, lm < 0 ? 0 : lm);
        if (lp > WAVE - 1) vn = 0.0;
        if (lm < 0) wp = 0.0;
      }
      const double sg = (L == 0) ? m.sig0[j] : 1.0;
      x[j] = sg * x[j] + vn + wp;
    }
  }
  // leaf pre-elimination x_tg -= leafm r_dg
  rdgb -= m.u->leafm * readlane(x[0], L_TG);
  if (lane == L_DG) x[0] += rdgb;
}

// x <- W^{-T} x (transpose of wsolve); a call, so that the step factors stay
// in memory rather than in registers across the reverse stage loop
template <int NS>
DEB_OUTLINE void wsolveT(const Mode<NS> &m, double (&xio)[NS]) {
  const int lane = lane_id();
  // a private copy (stores through xio could alias m for the compiler)
  double x[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) x[s] = xio[s];
  const double kba = readlane(x[0], L_A), kb1 = readlane(x[0], L_AHP);
  if (lane == L_A || lane == L_AHP) x[0] = 0.0;
  const double r1b = m.u->gh * kb1;
  double kab = kba + m.u->gh * m.u->J1a * kb1;
  const double c1kb = m.u->gh * kb1;
  double part[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    part[0] += m.Z[0][s] * x[s];
    part[1] += m.Z[1][s] * x[s];
    part[2] += m.Z[2][s] * x[s];
  }
  wave_sum4(part);
  double tt[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) tt[r] = m.u->c1Z[r] * c1kb + part[r];
  double gb[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) gb[c] = m.u->Sinv[0][c] * tt[0] + m.u->Sinv[1][c] * tt[1] + m.u->Sinv[2][c] * tt[2];
#pragma unroll
  for (int s = 0; s < NS; ++s)
    x[s] += m.Cf[0][s] * gb[0] + m.Cf[1][s] * gb[1] + m.Cf[2][s] * gb[2] + m.c1[s] * c1kb;
  bsolveT<NS>(m, x);
  double pj = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s) pj += m.jcol[s] * x[s];
  kab += wave_sum1(pj);
  if (lane == L_A) x[0] = m.u->inv_kaden * kab;
  if (lane == L_AHP) x[0] = r1b;
#pragma unroll
  for (int s = 0; s < NS; ++s) xio[s] = x[s];
}

// ---------------------------------------------------------------------------
// right-hand side contractions

// ---------------------------------------------------------------------------
// First-order contraction through background features.
//
// Every coefficient of row_visit depends on (a, theta) only through a few
// wave-uniform features (aH, 1/aH, opac, cs2, pb43, the density weights
// grhom Omega_c / a, ..., w, c_a^2, cs2_DE, a itself, a m_nu) and, for
// massive-nu rows, the bin velocity v_q = (1 + (a amnu / q)^2)^(-1/2), whose
// partials are folded into those of a and amnu.  The derivative of
// sum_rows sum_fields mul * coef is therefore sum_m Fbar_m dF_m, where Fbar_m
// (plain doubles) are the partials of the row formulas below and dF_m the
// features' tangents.
enum : int {
  FT_A = 0, FT_AH, FT_IAH, FT_OPAC, FT_CS2, FT_PB43, FT_RC, FT_RB, FT_RG, FT_RR, FT_RN, FT_RQ, FT_W, FT_CA2,
  FT_CS2Q, FT_AMNU, FT_N
};

template <class T>
__device__ __forceinline__ void features_of(const Ctx &cx, T a, const Bg<T> &b, T (&F)[FT_N]) {
  using P = ParT<T>;
  const P grhom = cv<T>(cx, F_GRHOM), grhog = cv<T>(cx, F_GRHOG), grhor = cv<T>(cx, F_GRHOR);
  const P Omegam = cv<T>(cx, F_OMEGAM), Omegab = cv<T>(cx, F_OMEGAB), OmegaDE = cv<T>(cx, F_OMEGADE);
  const P Neff = cv<T>(cx, F_NEFF), Nmnu = cv<T>(cx, F_NMNU);
  const T a2 = a * a;
  F[FT_A] = a;
  F[FT_AH] = b.aH;
  F[FT_IAH] = 1.0 / b.aH;
  F[FT_OPAC] = b.opac;
  F[FT_CS2] = b.cs2;
  F[FT_PB43] = b.pb43;
  F[FT_RC] = grhom * (Omegam - Omegab) / a;
  F[FT_RB] = grhom * Omegab / a;
  F[FT_RG] = grhog / a2;
  F[FT_RR] = grhor * Neff / a2;
  F[FT_RN] = grhor * Nmnu / a2;
  F[FT_RQ] = grhom * OmegaDE * b.rhoQ * a2;
  F[FT_W] = b.w;
  F[FT_CA2] = b.ca2;
  F[FT_CS2Q] = tconst<T>(0.0) + cv<T>(cx, F_CS2DE);
  F[FT_AMNU] = tconst<T>(0.0) + cv<T>(cx, F_AMNU);
}

template <class T>
__device__ __forceinline__ void features_t(Ctx &cx, T a, T (&F)[FT_N]) {
  const Bg<T> b = background<T>(cx, a);
  features_of<T>(cx, a, b, F);
}

// the features from the right-hand side's background (background_row), in
// plain doubles or along a
template <class T>
__device__ __forceinline__ void features_row(const Ctx &cx, const BgCache &g, const BgRow<T> &b, T (&F)[FT_N]) {
  const deb_cosmo_t &c = *cx.c;
  const T w = g.w0 + g.wa * (1.0 - b.a);
  F[FT_A] = b.a;
  F[FT_AH] = b.aH;
  F[FT_IAH] = b.iaH;
  F[FT_OPAC] = b.opac;
  F[FT_CS2] = b.cs2;
  F[FT_PB43] = g.pb * b.ia;
  F[FT_RC] = (c.grhom * (c.Omegam - c.Omegab)) * b.ia;
  F[FT_RB] = (c.grhom * c.Omegab) * b.ia;
  F[FT_RG] = c.grhog * b.ia2;
  F[FT_RR] = (c.grhor * c.Neff) * b.ia2;
  F[FT_RN] = g.gn * b.ia2;
  F[FT_RQ] = g.gde * b.rhoQ * (b.a * b.a);
  F[FT_W] = w;
  F[FT_CA2] = w + (g.wa * (1.0 / 3.0)) * (b.a * rcp_a(1.0 + w + 1e-6));
  F[FT_CS2Q] = tconst<T>(g.cs2Q);
  F[FT_AMNU] = tconst<T>(c.amnu);
}

// the mode's background at a; the spline windows go back to memory only when
// they have moved
template <int NS, class T>
__device__ __forceinline__ BgRow<T> mode_background(Mode<NS> &m, BgCache &g, T a) {
  g = m.bg;
  const double lo = g.xlo, hi = g.xhi;
  const BgRow<T> b = background_row(g, a);
  if (__ballot(!(lo == g.xlo && hi == g.xhi)) != 0) m.bg = g;
  return b;
}

// Values of the functionals of Y and of the "where they enter" sums of w that
// the first-order contraction below needs, plus (optionally) the transposed
// right-hand side A(a)^T w -- one plain-double pass over the rows.
template <class T>
struct RowSumsT {
  T H, E, Pi, F1;  // sum c_{h,eta,pi,1} Y
  T sh, se, sp;    // sum u_{h,eta,pi} w
};
using RowSums = RowSumsT<double>;

template <int NS>
__device__ __forceinline__ RowSums coef_pass_body(const RowK<NS> &K, const BgCache &g, const BgRow<double> &b,
                                                  double invtau, const double (&w)[NS], const double (&Y)[NS],
                                                  double (&out)[NS]) {
  const int lane = lane_id();
  double o[NS];
  double part[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  double cc[4][NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const Coef<double> r = row_lin<NS, double>(K, s, b, g, invtau);
    part[0] += r.ch * Y[s];
    part[1] += r.ceta * Y[s];
    part[2] += r.cpi * Y[s];
    part[3] += r.c1 * Y[s];
    part[4] += r.uh * w[s];
    part[5] += r.ueta * w[s];
    part[6] += r.upi * w[s];
    o[s] = r.diag * w[s] + from_next(r.sub * w[s]) + from_prev(r.sup * w[s]);
    if (s == 0) {
      const double lw = r.leaf * w[0];
      const double l_dg = readlane(lw, L_DG), l_tg = readlane(lw, L_TG);
      if (lane == L_TG) o[0] += l_dg;
      if (lane == L_DG) o[0] += l_tg;
    }
    cc[0][s] = r.ch;
    cc[1][s] = r.ceta;
    cc[2][s] = r.cpi;
    cc[3][s] = r.c1;
  }
  wave_sum8(part);
  RowSums rs{part[0], part[1], part[2], part[3], part[4], part[5], part[6]};
  const double wahp = readlane(w[0], L_AHP);
#pragma unroll
  for (int s = 0; s < NS; ++s) out[s] = o[s] + cc[0][s] * rs.sh + cc[1][s] * rs.se + cc[2][s] * rs.sp + cc[3][s] * wahp;
  return rs;
}
// the same as a call, with the features at a (the operator's test hook)
template <int NS>
DEB_OUTLINE RowSums coef_pass(Mode<NS> &m, Ctx &cx, double a, double invtau, const double (&w_in)[NS],
                              const double (&Y_in)[NS], double (&out)[NS], double (&fv_out)[FT_N]) {
  const RowK<NS> K = m.rk;
  BgCache g;
  double w[NS], Y[NS], o[NS], F[FT_N];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    w[s] = w_in[s];
    Y[s] = Y_in[s];
  }
  const BgRow<double> b = mode_background<NS>(m, g, a);
  const RowSums rs = coef_pass_body<NS>(K, g, b, invtau, w, Y, o);
  features_row(cx, g, b, F);
#pragma unroll
  for (int s = 0; s < NS; ++s) out[s] = o[s];
#pragma unroll
  for (int q = 0; q < FT_N; ++q) fv_out[q] = F[q];
  return rs;
}

// First-order contraction of S = sum_rows w_row f_row(a, Y): its partials with
// respect to the features, wave-uniform, for K contractions at once (fv[q] the
// feature values of contraction q).  The functionals (h', eta', Pi, f_1) enter
// through their values in rs, which is exact at first order: d(u H) = du H +
// u dH with dH = sum_rows dc_h Y, so sum_rows w u dH = s_h sum_rows dc_h Y.
//
// Only four partials need the lanes: the opacity, the massive and massless
// neutrino densities and the bin velocities (their -x dv/dx, x = a m_nu / q,
// carries both the a and the m_nu partial).  c_h is proportional to 1/aH and
// c_1 to a on every row, so those partials are s_h H and w_{ah'} f_1 over the
// feature; the remaining rows sit on fixed lanes of slot 0 and are combined as
// wave-uniform values read from there.  (Summed as 16 features per contraction
// from per-row multipliers, a stage's two contractions took 2400 instructions;
// this form takes about 700: gradient of 256 k at lmax 32 132 -> 108 ms.)
template <int NS, int K, class T = double>
__device__ __forceinline__ void feature_totals(const Ctx &cx, const RowK<NS> &R, const uint32_t (&rd)[NS],
                                               const T (&fv)[K][FT_N], const double (&Y)[K][NS],
                                               const double (&w)[K][NS], const RowSumsT<T> (&rs)[K],
                                               T (&fb)[K][FT_N]) {
  constexpr int C = ncomp<T>::value;
  static_assert(4 * K * C <= 8, "four lane sums per contraction");
  const double k2 = cx.k * cx.k, ik2 = 1.0 / k2, hk2 = 0.5 * ik2;
  T acc[K][4];  // opacity, velocity, massive and massless nu density
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const T *F = fv[q];
    const double wahp = readlane(w[q][0], L_AHP);
    const T shi = rs[q].sh * F[FT_IAH], wa = wahp * F[FT_A];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[q][i] = tconst<T>(0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const double y = Y[q][s], ws = w[q][s], ndy = R.nd[s] * y, ney = R.ne[s] * y;
      acc[q][0] = acc[q][0] + ws * (R.upi[s] * rs[q].Pi - R.ph[s] * y);
      if ((R.qmask >> s) & 1u) {
        T v, iv;
        bin_velocity(F[FT_A], R.aq[s], v, iv);
        const T x = F[FT_A] * R.aq[s];
        const double base = ws * (from_prev(y) * R.sub[s] + from_next(y) * R.sup[s]);
        const T g = ndy * (shi * iv - wa * (iv + v)) + ney * rs[q].se;
        const T vb = base - ndy * (F[FT_RN] * (shi * (iv * iv) + wa * (1.0 - iv * iv)));
        const bool qrow = rd_type(rd[s]) >= R_Q0 && rd_type(rd[s]) <= R_QLMAX;
        acc[q][1] = acc[q][1] - vb * ((x * x) * (v * v * v));
        acc[q][2] = acc[q][2] + sel(qrow, g, tconst<T>(0.0));
        acc[q][3] = acc[q][3] + sel(qrow, tconst<T>(0.0), g);
      } else {
        acc[q][3] = acc[q][3] + (ndy * (shi - 2.0 * wa) + ney * rs[q].se);
      }
    }
  }
  double flat[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) flat[i] = i < 4 * K * C ? comp(acc[(i / C) / 4 % K][(i / C) % 4], i % C) : 0.0;
  wave_sum8(flat);
#pragma unroll
  for (int i = 0; i < 4 * K * C; ++i) comp(acc[(i / C) / 4][(i / C) % 4], i % C) = flat[i];
  const double amnu = vval(fv[0][FT_AMNU]), iam = amnu != 0.0 ? 1.0 / amnu : 0.0;
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const T *F = fv[q];
    T *o = fb[q];
    auto y = [&](int lane) { return readlane(Y[q][0], lane); };
    auto W = [&](int lane) { return readlane(w[q][0], lane); };
    const T sh = rs[q].sh, se = rs[q].se;
    const T ia = rcp_a(F[FT_A]);
    const double wahp = W(L_AHP), wA = W(L_A), wtb = W(L_TB);
    const double ytb = y(L_TB), ytg = y(L_TG), ytc = y(L_TC);
    const T shi = sh * F[FT_IAH], wa = wahp * F[FT_A];
    const double d = wtb * (ytg - ytb);  // theta_b: pb43 opac on the super- minus the diagonal
    o[FT_OPAC] = acc[q][0] + (W(L_TG) * ytb + d * F[FT_PB43]);
    o[FT_PB43] = d * F[FT_OPAC];
    o[FT_CS2] = tconst<T>(wtb * y(L_DB) * k2);
    o[FT_RN] = acc[q][2];
    o[FT_RR] = acc[q][3];
    o[FT_RC] = y(L_DC) * (shi - wa) + (hk2 * ytc) * se;
    o[FT_RB] = y(L_DB) * (shi - wa) + (hk2 * ytb) * se;
    o[FT_RG] = y(L_DG) * (shi - 2.0 * wa) + ((4.0 / 3.0) * hk2 * ytg) * se;
    o[FT_IAH] = sh * rs[q].H * F[FT_AH];
    o[FT_A] = (acc[q][1] + wahp * rs[q].F1) * ia + wA * F[FT_AH];  // the a-row is aH a
    o[FT_AMNU] = acc[q][1] * iam;
    o[FT_AH] = wA * F[FT_A] - (W(L_TC) * ytc + wtb * ytb);
    o[FT_RQ] = tconst<T>(0.0);
    o[FT_W] = tconst<T>(0.0);
    o[FT_CA2] = tconst<T>(0.0);
    o[FT_CS2Q] = tconst<T>(0.0);
    if (!cx.lambda) {
      const T aH = F[FT_AH], cs2Q = F[FT_CS2Q], RQ = F[FT_RQ];
      const T opw = 1.0 + F[FT_W], dc = cs2Q - F[FT_CA2];
      const double yq = y(L_DQ), yt = y(L_TQ), wq = W(L_DQ), wt = W(L_TQ);
      const double dgq = wq * yq, sup = wq * yt, sub = wt * yq, dgt = wt * yt;
      const T ce = yt * se, c1q = yq * wa, c1t = (9.0 * ik2) * (yt * wa);  // c1 multipliers times a, and 9 / k^2
      const T g9 = (9.0 * ik2) * (aH * aH), t3 = 1.0 + 3.0 * cs2Q;
      const T iopw = rcp_a(opw), sk = (sub * k2) * iopw;
      const T og = opw * g9 * sup + c1t * (aH * opw * RQ);
      // diag -3 (cs2Q - w) aH, sup -opw - 9 opw (cs2Q - ca2) aH^2 / k^2, uh -opw / 2, ch RQ / aH,
      // c1 -a RQ (1 + 3 cs2Q); sub cs2Q k^2 / opw, diag -(1 - 3 cs2Q) aH, ceta opw RQ / 2 k^2,
      // c1 -9 a (cs2Q - ca2) aH opw RQ / k^2
      o[FT_CS2Q] = (3.0 * (dgt - dgq)) * aH - og - 3.0 * (c1q * RQ) + sk;
      o[FT_CA2] = og;
      o[FT_W] = (3.0 * dgq) * aH - sup - dc * (sup * g9 + c1t * (aH * RQ)) - (0.5 * wq) * rs[q].H - sk * cs2Q * iopw +
                hk2 * (ce * RQ);
      o[FT_AH] = o[FT_AH] - (3.0 * dgq) * (cs2Q - F[FT_W]) - dgt * (1.0 - 3.0 * cs2Q) -
                 opw * dc * ((18.0 * ik2 * sup) * aH + c1t * RQ);
      o[FT_RQ] = yq * shi - c1q * t3 + hk2 * (ce * opw) - c1t * (dc * aH * opw);
    }
  }
}

// One tangent direction per lane: lane & 7 == 0 carries d/da (component 0 of
// TL, seeded by seed_tl), lane & 7 == c (1 <= c <= ndir) the input tangent
// c - 1 (component 1, loaded through lane_ctx); TL arithmetic then costs
// three doubles per value instead of 2 + MAXDIR.  Only wave-uniform
// quantities may be computed in TL (a lane sum would mix directions).
using TL = dn<2>;

__device__ __forceinline__ Ctx lane_ctx(const Ctx &cx) {
  Ctx cl = cx;
  const int c = lane_id() & 7;
  const bool on = c >= 1 && c <= cx.ndir;
  cl.ndir = on ? 1 : 0;
  cl.dcos = cx.dcos + (on ? (c - 1) * COSMO_DOUBLES : 0);
  cl.dtab = cx.dtab + (on ? (c - 1) * cx.stride : 0);
  return cl;
}

__device__ __forceinline__ TL seed_tl(double a) {
  TL r;
  r = a;
  r.d[0] = (lane_id() & 7) == 0 ? 1.0 : 0.0;
  return r;
}

// the lane's direction of sum_m F_m fbs_m (fbs wave-uniform)
__device__ __forceinline__ double lane_dot(const TL (&F)[FT_N], const double (&fbs)[FT_N]) {
  double g = 0.0;
#pragma unroll
  for (int m = 0; m < FT_N; ++m) g += (F[m].d[0] + F[m].d[1]) * fbs[m];
  return g;
}

// feature values at a (plain doubles), wave-uniform: stored once per wave in
// LDS (every lane writes the same values)
template <int NS>
DEB_OUTLINE void feature_values(Mode<NS> &m, Ctx &cx, double a, lds_double *fv) {
  BgCache g;
  const BgRow<double> b = mode_background<NS>(m, g, a);
  double f[FT_N];
  features_row(cx, g, b, f);
#pragma unroll
  for (int q = 0; q < FT_N; ++q) fv[q] = f[q];
}

// the lane's direction of sum_m F_m(a) fbs_m (fbs wave-uniform): d/da on
// lanes with lane & 7 == 0, d/dtheta_{c-1} on lanes with lane & 7 == c
DEB_OUTLINE double lane_contract(const Ctx &cx, double a, const double (&fbs)[FT_N]) {
  Ctx cl = lane_ctx(cx);
  TL F[FT_N];
  features_t<TL>(cl, seed_tl(a), F);
  return lane_dot(F, fbs);
}

// The input-tangent directions of sum_m F_m(a_i) fbs_im for the eight stages
// of a reverse step at once: lane l evaluates the features at stage l >> 3's
// a along direction (l & 7) - 1 (none on l & 7 == 0).  cst: the stages' a_i
// (8 doubles), then their wave-uniform partials fbs_i (8 x FT_N).
DEB_OUTLINE double lane_contract_stages(const Ctx &cx, const lds_double *cst) {
  Ctx cl = lane_ctx(cx);
  const int i = lane_id() >> 3;
  TL as;
  as = (double)cst[i];
  TL F[FT_N];
  features_t<TL>(cl, as, F);
  double g = 0.0;
#pragma unroll
  for (int m = 0; m < FT_N; ++m) g += F[m].d[1] * (double)cst[8 + i * FT_N + m];
  return g;
}

// The a-column pass of the reverse step in dual arithmetic along a, with one
// background evaluation for all of it: out = A(a)^T w for the y-linear part of
// f (rows other than a; the a-column and the a-row go through the features)
// and its a-derivative; then, for S = sum_rows w f_row(a, Y), the functional
// sums and the per-lane feature partials P (fb.v) with their a-derivatives Q
// (fb.d), at the features of a.
template <int NS>
DEB_OUTLINE void acol_pass(Mode<NS> &m, Ctx &cx, dual a, double invtau, const double (&w_in)[NS],
                           const double (&Y_in)[NS], dual (&out_io)[NS], dual (&fb_out)[FT_N]) {
  using T = dual;
  const int lane = lane_id();
  double w[NS], Y[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    w[s] = w_in[s];
    Y[s] = Y_in[s];
  }
  const RowK<NS> K = m.rk;
  BgCache g;
  const BgRow<T> b = mode_background<NS>(m, g, a);
  T F[1][FT_N];
  features_row(cx, g, b, F[0]);
  T out[NS], part[7], cc[4][NS];
#pragma unroll
  for (int i = 0; i < 7; ++i) part[i] = tconst<T>(0.0);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const Coef<T> r = row_lin<NS, T>(K, s, b, g, invtau);
    T sw = r.sub * w[s];
    T pw = r.sup * w[s];
    out[s] = r.diag * w[s] + t_from_next(sw) + t_from_prev(pw);
    if (s == 0) {
      T lw = r.leaf * w[0];
      T l_dg = t_readlane(lw, L_DG), l_tg = t_readlane(lw, L_TG);
      if (lane == L_TG) out[0] = out[0] + l_dg;
      if (lane == L_DG) out[0] = out[0] + l_tg;
    }
    part[0] = part[0] + r.ch * Y[s];
    part[1] = part[1] + r.ceta * Y[s];
    part[2] = part[2] + r.cpi * Y[s];
    part[3] = part[3] + r.c1 * Y[s];
    part[4] = part[4] + r.uh * w[s];
    part[5] = part[5] + r.ueta * w[s];
    part[6] = part[6] + r.upi * w[s];
    cc[0][s] = r.ch;
    cc[1][s] = r.ceta;
    cc[2][s] = r.cpi;
    cc[3][s] = r.c1;
  }
  t_wave_sum<T, 7>(part);
  const double wahp = readlane(w[0], L_AHP);
#pragma unroll
  for (int s = 0; s < NS; ++s)
    out_io[s] = out[s] + cc[0][s] * part[4] + cc[1][s] * part[5] + cc[2][s] * part[6] + cc[3][s] * wahp;
  const RowSumsT<T> rs[1] = {RowSumsT<T>{part[0], part[1], part[2], part[3], part[4], part[5], part[6]}};
  double Yd[1][NS], wd[1][NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    Yd[0][s] = Y[s];
    wd[0][s] = w[s];
  }
  T fb[1][FT_N];
  feature_totals<NS, 1, T>(cx, K, m.rd, F, Yd, wd, rs, fb);
#pragma unroll
  for (int q = 0; q < FT_N; ++q) fb_out[q] = fb[0][q];
}

// Second order along one direction per lane: with P_m = dS/dF_m and
// Q_m = dP_m/da (wave-uniform) for S(F(a, theta)), returns on lane direction c
// d/dc (dS/da) = sum_m Q_m dF_m/dc + P_m d2F_m/(da dc)  (c = a on lane & 7 == 0).
// PQ: P (FT_N doubles), then Q, one copy per wave in LDS.  Features in nested
// duals: outer component along the lane's direction, inner along a.
using TL2 = dn<2, dual>;
DEB_OUTLINE double lane_contract2(const Ctx &cx, double a, const lds_double *PQ) {
  Ctx cl = lane_ctx(cx);
  TL2 as;
  as = a;
  as.v.d = 1.0;
  as.d[0].v = (lane_id() & 7) == 0 ? 1.0 : 0.0;
  TL2 F[FT_N];
  features_t<TL2>(cl, as, F);
  double g = 0.0;
#pragma unroll
  for (int m = 0; m < FT_N; ++m)
    g += (double)PQ[FT_N + m] * (F[m].d[0].v + F[m].d[1].v) + (double)PQ[m] * (F[m].d[0].d + F[m].d[1].d);
  return g;
}

// the lane-direction result of every direction: out[j] = d/dtheta_j
__device__ __forceinline__ void lane_gather(double g, int ndir, double (&out)[MAXDIR]) {
#pragma unroll
  for (int j = 0; j < MAXDIR; ++j) out[j] = j < ndir ? readlane(g, j + 1) : 0.0;
}

// row sums of the step Jacobian J(t0, y0) kept by the factorisation
template <int NS>
__device__ __forceinline__ RowSums jac_sums(const Mode<NS> &m, const double (&Y)[NS], const double (&w)[NS]) {
  double part[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    part[0] += m.Cf[0][s] * Y[s];
    part[1] += m.Cf[1][s] * Y[s];
    part[2] += m.Cf[2][s] * Y[s];
    part[3] += m.c1[s] * Y[s];
    part[4] += m.U[0][s] * w[s];
    part[5] += m.U[1][s] * w[s];
    part[6] += m.U[2][s] * w[s];
  }
  wave_sum8(part);
  return RowSums{part[0], part[1], part[2], part[3], part[4], part[5], part[6]};
}

// (Bound by the latency of the step factors and row constants in the caller's
// frame and by instruction issue.  With the rows from the mode's constants and
// one background evaluation for rows and features the gradient of 256 k at lmax
// 32 went from 160 to 136 ms; inlined into the stage loop it measured 133 ms
// where the call takes 112.)
// The row work of one reverse stage as a single call: the transposed row pass
// at the stage point (ub = J(t_i, u_i)^T rb, the stage's features and their
// a-derivative dfa), the row sums of the J(t0, y0) k_i term, and the feature
// partials of both contractions, each summed over the wave: the J-term's (at
// the features fvJ of a0, multipliers without the a-row) accumulated into fbJ,
// the stage's stored to fb_out and contracted with dfa into the a-direction of
// ub (fbJ and fb_out: one copy per wave in LDS).
template <int NS>
DEB_OUTLINE void stage_rows(Ctx &cx, Mode<NS> &m, double ai, double iti, const double (&rb_in)[NS],
                            const double (&u_in)[NS], const double (&ki_in)[NS], const lds_double *fvJ_in,
                            double (&ub_out)[NS], lds_double *fbJ_io, lds_double *fb_out) {
  const int lane = lane_id();
  double rb[NS], u[NS], ki[NS], ub[NS], dfa[FT_N];
  double fvs[2][FT_N], fbs[2][FT_N];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    rb[s] = rb_in[s];
    u[s] = u_in[s];
    ki[s] = ki_in[s];
  }
#pragma unroll
  for (int q = 0; q < FT_N; ++q) {
    fvs[1][q] = (double)fvJ_in[q];
  }
  // one background evaluation along a: its values for the rows, both for the features
  RowSums rsq[2];
  const RowK<NS> K = m.rk;
  {
    BgCache g;
    const BgRow<dual> bd = mode_background<NS>(m, g, mkd(ai, 1.0));
    dual F[FT_N];
    features_row(cx, g, bd, F);
#pragma unroll
    for (int q = 0; q < FT_N; ++q) {
      fvs[0][q] = F[q].v;
      dfa[q] = F[q].d;
    }
    const BgRow<double> b{bd.a.v, bd.aH.v, bd.iaH.v, bd.ia.v, bd.ia2.v, bd.opac.v, bd.cs2.v, bd.po.v, bd.rhoQ.v};
    rsq[0] = coef_pass_body<NS>(K, g, b, iti, rb, u, ub);
  }
  double Yq[2][NS], wq[2][NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    Yq[0][s] = u[s];
    wq[0][s] = rb[s];
    Yq[1][s] = ki[s];
    wq[1][s] = (s == 0 && lane == L_A) ? 0.0 : rb[s];
  }
  rsq[1] = jac_sums<NS>(m, ki, wq[1]);
  feature_totals<NS, 2>(cx, K, m.rd, fvs, Yq, wq, rsq, fbs);
  double ga = 0.0;
#pragma unroll
  for (int q = 0; q < FT_N; ++q) ga += dfa[q] * fbs[0][q];
  if (lane == L_A) ub[0] += ga;
#pragma unroll
  for (int s = 0; s < NS; ++s) ub_out[s] = ub[s];
#pragma unroll
  for (int q = 0; q < FT_N; ++q) {
    fb_out[q] = fbs[0][q];
    fbJ_io[q] += fbs[1][q];
  }
}

__device__ __forceinline__ TD seed_td(double v, double d0) {
  TD r;
  r = v;
  r.d[0] = d0;
  return r;
}

// one forward step from (t0, y0) to y1, its eight stage vectors stored in
// K[8][NS][64]
template <int NS>
__device__ __forceinline__ void step_store(Mode<NS> &m, double t0, double h, const double (&y0)[NS],
                                           double (&y1)[NS], double *K, lds_double *kl) {
  const int lane = lane_id();
  double err[NS];
  auto store = [&](int i, const double (&k)[NS]) {
#pragma unroll
    for (int s = 0; s < NS; ++s) K[(i * NS + s) * WAVE + lane] = k[s];
  };
  rodas5_step_s<NS>(m, t0, h, y0, y1, err, store, kl);
}

// ---------------------------------------------------------------------------
// reverse of one Rodas5 step.  In: ybar = dL/dy1.  Out: ybar = dL/dy0,
// tbar += dL/dt0 (h fixed), hbar += dL/dh, thb[j] += dL/dtheta_j (wave-uniform).
// K: the step's eight stage vectors ([8][NS][64], written by step_store);
// KBl: per-wave LDS scratch of 7 stage vectors.  The factorisation of W at
// (t0, y0) is recomputed into m.
template <int NS>
__device__ __forceinline__ void rodas5_step_vjp(Mode<NS> &m, Ctx &cx, double t0, double h,
                                                const double (&y0)[NS], double (&ybar)[NS], double (&thb)[MAXDIR],
                                                double &tbar, double &hbar, const double *K, double *KBl) {
  const int lane = lane_id();
  auto Kp = [&](int i, int s) -> double { return K[(i * NS + s) * WAVE + lane]; };
  auto KBp = [&](int i, int s) -> double & { return KBl[(i * NS + s) * WAVE + lane]; };
  // per stage: its a and its wave-uniform feature partials (written by every
  // lane alike)
  __shared__ double cst_[8 * (1 + FT_N)];
  lds_double *const cst = (lds_double *)cst_;
  factor_call<NS>(m, t0, y0, h);
  // explicit tau dependence (hierarchy truncations): d f_row / d tau = tw / tau^2 * y_row
  double tw[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) tw[s] = m.rk.tr[s];
  const double it0 = 1.0 / t0;
  const double a0 = readlane(y0[0], L_A);
  double dT[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) dT[s] = tw[s] * it0 * it0 * y0[s];
  const double gamma = R5::gamma;
  const double ih = 1.0 / h;
  double y1b[NS], y0b[NS], dTb[NS], rho[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    y1b[s] = ybar[s];
    y0b[s] = ybar[s];  // y1 = y0 + sum A8 k
    dTb[s] = 0.0;
    rho[s] = 0.0;
  }
#pragma unroll
  for (int j = 0; j < 7; ++j)
#pragma unroll
    for (int s = 0; s < NS; ++s) KBp(j, s) = kA8[j] * y1b[s];
  double th_acc[MAXDIR];
#pragma unroll
  for (int j = 0; j < MAXDIR; ++j) th_acc[j] = 0.0;
  double a0b = 0.0, t0b = 0.0, hb = 0.0;
  // Feature partials, one row pass per stage (stage_rows) with two
  // contractions: f(t_i, u_i) at the stage's features (contracted every
  // stage) and the J(t0, y0) k_i term at the features fvJ of a0 (its partials
  // fbJ accumulate over the stages and are contracted once).
  // the features of a0 and the J-term's partials (summed over the wave) are
  // wave-uniform: one copy per wave in LDS (written by every lane alike)
  __shared__ double fvJ_[FT_N], fbJ_[FT_N];
  lds_double *const fvJ = (lds_double *)fvJ_, *const fbJl = (lds_double *)fbJ_;
  feature_values<NS>(m, cx, a0, fvJ);
#pragma unroll
  for (int q = 0; q < FT_N; ++q) fbJl[q] = 0.0;
#pragma nounroll
  for (int i = 7; i >= 0; --i) {
    double rb[NS], ki[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) rb[s] = (i == 7) ? y1b[s] * kA8[7] : KBp(i, s);
    wsolveT<NS>(m, rb);
    // stage point u_i and the combination sum_j C_ij k_j
    double u[NS], ck[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      u[s] = y0[s];
      ck[s] = 0.0;
    }
    // this stage's vector and the earlier ones in one batch of loads (the
    // tableau's rows are zero from column i on, so the sums add exact zeros
    // there; stages 1 to 4 leave the last four columns out)
    {
      double kj[7][NS];
#pragma unroll
      for (int j = 0; j < 7; ++j)
#pragma unroll
        for (int s = 0; s < NS; ++s) kj[j][s] = (j < 3 || i > 3) ? Kp(j, s) : 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) ki[s] = Kp(i, s);
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        const double aij = kA[i][j], cij = kC[i][j];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          u[s] += aij * kj[j][s];
          ck[s] += cij * kj[j][s];
        }
      }
    }
    const double ti = t0 + kc[i] * h;
    const double iti = 1.0 / ti;
    // dot products: h-derivative of W, C/h and d h dT terms; explicit time
    // dependence at the stage point and of J at (t0, y0)
    double dots[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      dots[0] += rb[s] * (ki[s] / (gamma * h * h) - ck[s] * ih * ih + kd[i] * dT[s]);
      dots[1] += rb[s] * tw[s] * iti * iti * u[s];
      dots[2] += rb[s] * tw[s] * it0 * it0 * ki[s];
    }
    wave_sum4(dots);
    hb += dots[0] + kc[i] * dots[1];
    t0b += dots[1] + dots[2];
    if (kd[i] != 0.0) {
#pragma unroll
      for (int s = 0; s < NS; ++s) dTb[s] += kd[i] * h * rb[s];
    }
    // f(t_i, u_i): ubar = J(t_i, u_i)^T rbar, and the J(t0, y0) k_i term
    // (its y-linear part at a0; the a-column goes through rho)
    double ub[NS];
    {
      const double ai = readlane(u[0], L_A);
      stage_rows<NS>(cx, m, ai, iti, rb, u, ki, fvJ, ub, fbJl, cst + 8 + i * FT_N);
      cst[i] = ai;
      const double kia = readlane(ki[0], L_A);
#pragma unroll
      for (int s = 0; s < NS; ++s) rho[s] += kia * rb[s];
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) y0b[s] += ub[s];
    // cotangents of the earlier stages, in two batches (those of this stage on
    // have been read, and their tableau entries are zero)
    auto feed = [&](auto first, auto count) {
      constexpr int J0 = decltype(first)::value, NJ = decltype(count)::value;
      double kb[NJ][NS];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int s = 0; s < NS; ++s) kb[j][s] = KBp(J0 + j, s);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const double aij = kA[i][J0 + j], cij = kC[i][J0 + j] * ih;
#pragma unroll
        for (int s = 0; s < NS; ++s) KBp(J0 + j, s) = kb[j][s] + (cij * rb[s] + aij * ub[s]);
      }
    };
    feed(std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
    if (i > 3) feed(std::integral_constant<int, 3>{}, std::integral_constant<int, 4>{});
  }
  // the stages' input-tangent directions
  {
    const double g = lane_contract_stages(cx, cst);
#pragma unroll
    for (int j = 0; j < MAXDIR; ++j) {
      if (j < cx.ndir) {
        double t = 0.0;
#pragma unroll
        for (int st = 0; st < 8; ++st) t += readlane(g, st * 8 + j + 1);
        th_acc[j] += t;
      }
    }
  }
  // a-column of J(t0, y0): rho^T df/da, differentiated along y0, a0 and theta
  {
    dual ad;
    ad.v = a0;
    ad.d = 1.0;
    // rho^T A'(a) (the derivative of the transposed apply), and for
    // S = rho^T f(a, y0) the feature partials in dual arithmetic
    dual gy[NS], fbd[FT_N];
    acol_pass<NS>(m, cx, ad, it0, rho, y0, gy, fbd);
#pragma unroll
    for (int s = 0; s < NS; ++s) y0b[s] += gy[s].d;
    // the feature partials P and their a-derivative Q, kept in the stage block
    // (whose contraction has been read), then the features' second derivatives
    // (the J(t0, y0) k_i terms' partials join Q: contracted with the same
    // feature tangents at a0, to first order)
#pragma unroll
    for (int q = 0; q < FT_N; ++q) {
      cst[q] = fbd[q].v;
      cst[FT_N + q] = fbd[q].d + fbJl[q];
    }
    const double g = lane_contract2(cx, a0, cst);
    a0b += readlane(g, 0);
    double tl[MAXDIR];
    lane_gather(g, cx.ndir, tl);
#pragma unroll
    for (int j = 0; j < MAXDIR; ++j) th_acc[j] += tl[j];
  }
  // dT = D(t0) y0
  {
    double pt = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      y0b[s] += tw[s] * it0 * it0 * dTb[s];
      pt += dTb[s] * (-2.0 * tw[s] * it0 * it0 * it0) * y0[s];
    }
    t0b += wave_sum1(pt);
  }
  if (lane == L_A) y0b[0] += a0b;
#pragma unroll
  for (int s = 0; s < NS; ++s) ybar[s] = y0b[s];
#pragma unroll
  for (int j = 0; j < MAXDIR; ++j) thb[j] += th_acc[j];
  tbar += t0b;
  hbar += hb;
}

// ---------------------------------------------------------------------------
// start time and initial conditions in tangent arithmetic (the same formulas
// as start_time and initial_conditions)

template <class T>
__device__ __forceinline__ T start_time_t(Ctx &cx, T tau_out_min) {
  using P = ParT<T>;
  const P taumin = cv<T>(cx, F_TAUMIN), YHe = cv<T>(cx, F_YHE), Omegab = cv<T>(cx, F_OMEGAB), H0 = cv<T>(cx, F_H0);
  const T tau0 = taumin;
  const T tau1 = spl_at<T>(cx, DEB_SPL_TAU_A, tconst<T>(0.1));
  const double tau_k = 1.0 / cx.k;
  const P akthom = 2.3048e-9 * (1.0 - YHe) * Omegab * H0 * H0;
  T lt[2];
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    // the bisection compares signs only: the root's tangent flows through
    // the bracket end points
    T xl = dlog(tau0), xr = dlog(tau1);
    auto fn = [&](const T &x) {
      T tau = dexp(x);
      T a = spl_at<T>(cx, DEB_SPL_A_TAU, tau);
      Bg<T> b = background<T>(cx, a);
      if (which == 0) return vval((1.0 / b.aH) / tau_k / 0.07 - 1.0);
      T xe = spl_at<T>(cx, DEB_SPL_XE_TAU, tau);
      T opac = xe * akthom / (a * a);
      return vval((1.0 / opac) / (1.0 / b.aH) / 0.0004 - 1.0);
    };
    for (int i = 0; i < 7; ++i) {
      T xm = 0.5 * (xl + xr);
      if (fn(xm) * fn(xl) > 0) xl = xm; else xr = xm;
    }
    lt[which] = 0.5 * (xl + xr);
  }
  T ts = dexp(vval(lt[1]) < vval(lt[0]) ? lt[1] : lt[0]);
  return 0.99 * (vval(tau_out_min) < vval(ts) ? tau_out_min : ts);
}

template <int NS, class T>
__device__ __forceinline__ void ics_t(Ctx &cx, const uint32_t (&rd)[NS], T tau, T (&y)[NS]) {
  using P = ParT<T>;
  const P grhom = cv<T>(cx, F_GRHOM), grhog = cv<T>(cx, F_GRHOG), grhor = cv<T>(cx, F_GRHOR);
  const P Omegam = cv<T>(cx, F_OMEGAM), Omegab = cv<T>(cx, F_OMEGAB), Neff = cv<T>(cx, F_NEFF);
  const P Nmnu = cv<T>(cx, F_NMNU), amnu = cv<T>(cx, F_AMNU), w0 = cv<T>(cx, F_W0), wa = cv<T>(cx, F_WA);
  const P cs2Q = cv<T>(cx, F_CS2DE);
  const double k = cx.k;
  T a = spl_at<T>(cx, DEB_SPL_A_TAU, tau);
  T rnu = dexp(spl_at<T>(cx, DEB_SPL_LOGRHONU_LOGA, dlog(a)));
  T a4 = a * a * a * a;
  T rhom = grhom * Omegam / (a * a * a);
  T rhor = (grhog + grhor * (Neff + Nmnu * rnu)) / a4;
  T rhonu = grhor * (Neff + Nmnu * rnu) / a4;
  P fracb = Omegab / Omegam;
  T fracnu = rhonu / rhor;
  T om = a * rhom / dsqrt(rhor);
  const double C = -1.0;
  T kt = k * tau;
  T deltag = -(kt * kt) / 3.0 * (1.0 - om * tau / 5.0) * C;
  T thetag = -(kt * kt * kt) / tau / 36.0 *
             (1.0 - 3.0 * (1.0 + 5.0 * fracb - fracnu) / 20.0 / (1.0 - fracnu) * om * tau) * C;
  T thetar = -(kt * kt * kt * kt) / tau / 36.0 / (4.0 * fracnu + 15.0) *
             (4.0 * fracnu + 11.0 + 12.0 -
              3.0 * (8.0 * fracnu * fracnu + 50.0 * fracnu + 275.0) / 20.0 / (2.0 * fracnu + 15.0) * tau * om) * C;
  T shearr = (kt * kt) / (45.0 + 12.0 * fracnu) * 2.0 *
             (1.0 + (4.0 * fracnu - 5.0) / 4.0 / (2.0 * fracnu + 15.0) * tau * om) * C;
  T wQ = w0 + wa * (1.0 - a);
  T deltaq = (kt * kt) / 4.0 * (1.0 + wQ) * (4.0 - 3.0 * cs2Q) / (4.0 - 6.0 * wQ + 3.0 * cs2Q) * C;
  T thetaq = (kt * kt * kt * kt) / tau / 4.0 * cs2Q / (4.0 - 6.0 * wQ + 3.0 * cs2Q) * C;
  if (cx.lambda) {
    deltaq = tconst<T>(0.0);
    thetaq = tconst<T>(0.0);
  }
  T eta = C * (1.0 - (kt * kt) / 12.0 / (15.0 + 4.0 * fracnu) *
                         (5.0 + 4.0 * fracnu - (16.0 * fracnu * fracnu + 280.0 * fracnu + 325.0) / 10.0 /
                                                   (2.0 * fracnu + 15.0) * tau * om));
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const uint32_t t = rd_type(rd[s]);
    const int qi = (int)rd_q(rd[s]);
    T v = tconst<T>(0.0);
    switch (t) {
      case R_A: v = a; break;
      case R_ETA: v = eta; break;
      case R_DC: v = 0.75 * deltag; break;
      case R_DB: v = 0.75 * deltag; break;
      case R_TB: v = thetag; break;
      case R_DG: v = deltag; break;
      case R_TG: v = thetag; break;
      case R_DR: v = deltag; break;
      case R_TR: v = thetar; break;
      case R_FR2: v = 2.0 * shearr; break;
      case R_DQ: v = deltaq; break;
      case R_TQ: v = thetaq; break;
      case R_Q0: case R_Q1: case R_Q2: {
        T aq = a * amnu / cx.q[qi];
        T vq = 1.0 / dsqrt(1.0 + aq * aq);
        const double dl = cx.dlnf[qi];
        if (t == R_Q0) v = -0.25 * dl * deltag;
        else if (t == R_Q1) v = -dl * thetar / vq / k / 3.0;
        else v = -0.5 * dl * shearr;
        break;
      }
      default: break;
    }
    y[s] = v;
  }
}

// ---------------------------------------------------------------------------
// the gradient kernel's arguments
struct AdjArgs {
  int ndir;
  const double *dcos;     // [n_cosmo][ndir][24]
  const double *dtab;     // [n_cosmo][ndir][stride]
  const double *dtau;     // [n_cosmo][ndir][nout]
  const double *ybar;     // [n_cosmo][nk][nout][20]  dL/d(output fields)
  const int32_t *status;  // [n_cosmo][nk] of the taped forward solve
  double *grad;           // [n_cosmo][nk][ndir]
  TapeView tape;
  double *rings;          // [n_rings][ring_doubles(NS, C)] reverse-launch rings
  int32_t *ring_busy;     // [n_rings] 1 while a wave owns the ring
  const int32_t *order;   // [n_modes] launch order (mode indices, longest first), or null
  int n_rings;
  int n_in;               // state entries read by the output conversion
  int32_t in_idx[WAVE];   // their reference indices, one per lane
};

// reference indices of the state entries read by the output conversion, one
// per lane (host side: fills AdjArgs::in_idx)
inline int output_inputs(const deb_config_t &c, int32_t *idx) {
  const int lg = c.lmaxg, lgp = c.lmaxgp, lr = c.lmaxr, nq = c.nqmax;
  const int n = 12 + lg + lgp + lr + nq * (c.lmaxnu + 1);
  const int ir = 9 + lg + lgp, iq0 = 10 + lg + lgp + lr;
  int m = 0;
  for (int i : {0, 2, 3, 4, 5, 6, 7, 8}) idx[m++] = i;
  idx[m++] = ir;
  idx[m++] = ir + 1;
  for (int i = 0; i < nq; ++i) idx[m++] = iq0 + i;
  for (int i = 0; i < nq; ++i) idx[m++] = iq0 + nq + i;
  idx[m++] = n - 2;
  idx[m++] = n - 1;
  for (int i = m; i < WAVE; ++i) idx[i] = -1;
  return m;
}

// reverse of the output conversion of one output time: yb = dL/dy (slot
// layout), thb += dL/dtheta at fixed y.  w: the 20 field cotangents.
template <int NS>
__device__ __forceinline__ void output_vjp(const Params<NS> &P, Ctx &cx, const AdjArgs &A, const uint32_t (&rd)[NS],
                                           const double (&yo)[NS], const double *w, double *ls, double *lg,
                                           double (&yb)[NS], double (&thb)[MAXDIR]) {
  const int lane = lane_id();
  const int L0 = P.cfg.lmaxg, L1 = P.cfg.lmaxgp, L2 = P.cfg.lmaxr;
  for (int i = lane; i < P.n; i += WAVE) lg[i] = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (rd_type(rd[s]) != R_NONE) ls[rd_idx(rd[s])] = yo[s];
  BlockSync()();
  double om[DEB_NOUT_FIELDS];
#pragma unroll
  for (int f = 0; f < DEB_NOUT_FIELDS; ++f) om[f] = w[f];
  {
    TD acc = tconst<TD>(0.0);
    output_fields_t<TD>(cx, [&](int i) { return tconst<TD>(ls[i]); }, L0, L1, L2, P.nq, P.n,
                        [&](int f, const TD &v) { acc = acc + v * om[f]; });
#pragma unroll
    for (int j = 0; j < MAXDIR; ++j) thb[j] += acc.d[j + 1];
  }
  if (lane < A.n_in) {
    const int seed = A.in_idx[lane];
    dual acc;
    acc = 0.0;
    output_fields_t<dual>(cx,
                          [&](int i) {
                            dual r;
                            r.v = ls[i];
                            r.d = (i == seed) ? 1.0 : 0.0;
                            return r;
                          },
                          L0, L1, L2, P.nq, P.n, [&](int f, const dual &v) { acc = acc + v * om[f]; });
    lg[seed] = acc.d;
  }
  BlockSync()();
#pragma unroll
  for (int s = 0; s < NS; ++s) yb[s] = rd_type(rd[s]) != R_NONE ? lg[rd_idx(rd[s])] : 0.0;
  BlockSync()();
}

// one (cosmology, k) item of the gradient kernel.  ring: this wave's ring
// (ring_doubles(NS, C) doubles of device memory, owned for the item's life);
// KBl, ls, lg: per-wave LDS scratch; cx: the wave's context record, in LDS in
// the kernel (its fields are wave-uniform, so one copy serves the wave, and the
// row passes read it there instead of from a per-lane stack copy; every lane
// stores the same values into it)
template <int NS>
__device__ __forceinline__ void adjoint_mode(const Params<NS> &P, const AdjArgs &A, int ci, int ki, double *ring,
                                             double *KBl, double *ls, double *lg, lds_double *pcr, Ctx &cx) {
  const int lane = lane_id();
  const long long item = (long long)ci * P.nk + ki;
  double *gout = A.grad + item * A.ndir;
  if (A.status[item] != DEB_STATUS_OK || A.tape.count[item] < 2) {
    if (lane < A.ndir) gout[lane] = __builtin_nan("");
    return;
  }
  const double k = P.kmodes[item];
  make_ctx<NS>(cx, P, ci, k);
  cx.ndir = A.ndir;
  cx.dcos = A.dcos + (long long)ci * A.ndir * COSMO_DOUBLES;
  cx.dtab = A.dtab + (long long)ci * A.ndir * P.table_stride;
  __shared__ ModeU mu;
  Mode<NS> m;
  m.pcr = pcr;
  m.u = (lds_mode_u *)&mu;
#pragma unroll
  for (int s = 0; s < NS; ++s) m.rd[s] = P.rowdesc[s][lane];
  row_consts<NS>(m.rd, cx, m.rk);
  bg_init(cx, m.bg);
  m.nlev = mode_levels(P.cfg, P.nq);
  const double *tout = P.tau_out + (long long)ci * P.nout;
  const double *dtout = A.dtau + (long long)ci * A.ndir * P.nout;
  int imin = 0, imax = 0;
  for (int i = 1; i < P.nout; ++i) {
    if (tout[i] < tout[imin]) imin = i;
    if (tout[i] > tout[imax]) imax = i;
  }
  // the tape: N accepted steps in segments of C, the last segment's chunk
  // first (a chunk that holds only the final state, when C divides N, is skipped)
  const TapeView &tv = A.tape;
  const int C = tv.ckpt;
  const int N = tv.count[item] - 1;
  auto chunk_t = [&](long long c) { return reinterpret_cast<const double *>(tv.pool + c * tv.chunk_bytes + 64); };
  auto chunk_y = [&](long long c) { return reinterpret_cast<const double *>(tv.pool + c * tv.chunk_bytes + tv.state_off); };
  auto chunk_prev = [&](long long c) { return *reinterpret_cast<const long long *>(tv.pool + c * tv.chunk_bytes); };
  long long chunk = tv.last[item];
  int seg = N / C;
  if (N % C == 0) {
    chunk = chunk_prev(chunk);
    --seg;
  }
  double t0 = 0.0;  // the first state's time
  {
    long long c = chunk;
    for (int s2 = seg; s2 > 0; --s2) c = chunk_prev(c);
    t0 = chunk_t(c)[0];
  }
  auto ring_y = [&](int j) { return ring + (long long)j * NS * WAVE; };
  auto ring_k = [&](int j) { return ring + ((long long)(C + 1) + 8LL * j) * NS * WAVE; };
  const double T1 = tout[imax];
  const double span = T1 - t0;
  double thb[MAXDIR];
#pragma unroll
  for (int j = 0; j < MAXDIR; ++j) thb[j] = 0.0;
  double Tb0 = 0.0, Tb1 = 0.0;
  double yb[NS], pend[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) yb[s] = 0.0;
  const double *wbase = A.ybar + item * (long long)P.nout * DEB_NOUT_FIELDS;
  int iout = P.nout - 1;
  for (; seg >= 0; --seg, chunk = chunk_prev(chunk)) {
    const int nL = min(C, N - seg * C);
    const double *tt = chunk_t(chunk);
    // forward again over the segment from its checkpoint: states and stage
    // vectors into the ring
    {
      // the step factors of the recompute are its own: they stay in registers,
      // where those of the reversal live in memory across its calls
      Mode<NS> mr;
      mr.pcr = pcr;
      mr.u = (lds_mode_u *)&mu;
      mr.rk = m.rk;
      mr.bg = m.bg;
      mr.nlev = m.nlev;
      double y[NS], y1[NS];
      const double *yc = chunk_y(chunk);
#pragma unroll
      for (int s = 0; s < NS; ++s) y[s] = yc[s * WAVE + lane];
      for (int j = 0; j < nL; ++j) {
        double *ry = ring_y(j);
#pragma unroll
        for (int s = 0; s < NS; ++s) ry[s * WAVE + lane] = y[s];
        step_store<NS>(mr, tt[j], tt[j + 1] - tt[j], y, y1, ring_k(j), (lds_double *)KBl);
#pragma unroll
        for (int s = 0; s < NS; ++s) y[s] = y1[s];
      }
      double *ry = ring_y(nL);
#pragma unroll
      for (int s = 0; s < NS; ++s) ry[s * WAVE + lane] = y[s];
    }
    for (int j = nL - 1; j >= 0; --j) {
      const int n = seg * C + j;
      double ycur[NS], ynext[NS];
      {
        const double *r0 = ring_y(j), *r1 = ring_y(j + 1);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          ycur[s] = r0[s * WAVE + lane];
          ynext[s] = r1[s * WAVE + lane];
        }
      }
      const double tcur = tt[j];
      const double h = tt[j + 1] - tcur;
      double tb = 0.0, hb = 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) pend[s] = 0.0;
      // outputs interpolated inside this step (t_n < tau_o <= t_{n+1}; step 0
      // also takes tau_o <= t_1)
      while (iout >= 0 && (tout[iout] > tcur || n == 0)) {
        const double th = (tout[iout] - tcur) / h;
        double yo[NS], ybo[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) yo[s] = ycur[s] + th * (ynext[s] - ycur[s]);
        output_vjp<NS>(P, cx, A, m.rd, yo, wbase + (long long)iout * DEB_NOUT_FIELDS, ls, lg, ybo, thb);
        double pth = 0.0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          yb[s] += th * ybo[s];
          pend[s] += (1.0 - th) * ybo[s];
          pth += ybo[s] * (ynext[s] - ycur[s]);
        }
        const double thbar = wave_sum1(pth);
        const double taub = thbar / h;
#pragma unroll
        for (int jj = 0; jj < MAXDIR; ++jj)
          if (jj < A.ndir) thb[jj] += taub * dtout[jj * P.nout + iout];
        tb += -thbar / h;
        hb += -thbar * th / h;
        --iout;
      }
      rodas5_step_vjp<NS>(m, cx, tcur, h, ycur, yb, thb, tb, hb, ring_k(j), KBl);
#pragma unroll
      for (int s = 0; s < NS; ++s) yb[s] += pend[s];
      const double sn = (tcur - t0) / span, dsn = h / span;
      Tb0 += tb * (1.0 - sn) - hb * dsn;
      Tb1 += tb * sn + hb * dsn;
    }
  }
  // initial conditions y(t0) = IC(t0)
  {
    TD y0t[NS];
    ics_t<NS, TD>(cx, m.rd, seed_td(t0, 1.0), y0t);
    TD acc[1];
    acc[0] = tconst<TD>(0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[0] = acc[0] + y0t[s] * yb[s];
    t_wave_sum<TD, 1>(acc);
    Tb0 += acc[0].d[0];
#pragma unroll
    for (int j = 0; j < MAXDIR; ++j) thb[j] += acc[0].d[j + 1];
  }
  // t0 = start time(min tau_out), t1 = max tau_out
  {
    TD tmin;
    tmin = tout[imin];
#pragma unroll
    for (int j = 0; j < MAXDIR; ++j) tmin.d[j + 1] = j < A.ndir ? dtout[j * P.nout + imin] : 0.0;
    TD ts = start_time_t<TD>(cx, tmin);
#pragma unroll
    for (int j = 0; j < MAXDIR; ++j) {
      thb[j] += Tb0 * ts.d[j + 1];
      if (j < A.ndir) thb[j] += Tb1 * dtout[j * P.nout + imax];
    }
  }
#pragma unroll
  for (int j = 0; j < MAXDIR; ++j)
    if (lane == j && j < A.ndir) gout[j] = thb[j];
}

}  // namespace deb

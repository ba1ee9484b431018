// Per-mode physics and the structured Rodas5 step (device side).
//
// Physics: model_synchronous (src/discoeb/perturbations.py:84-371), written as
// one row per lane: f_row = sub*y[lane-1] + diag*y[lane] + sup*y[lane+1]
//   + uh*h' + ueta*eta' + upi*Pi + leaf*y[partner]
// with the metric functionals h', eta' (perturbations.py:257-260), the
// polarization source Pi = F_2 + G_0 + G_2 (:286) and the a*h' accumulator
// f_1 (:252) obtained as wave reductions sum(c * y).
#pragma once

#include <type_traits>

#include "deb_device.h"

namespace deb {

struct Ctx {
  const deb_cosmo_t *c;
  Spl sp[DEB_NSPLINE];
  double k;
  int nq;
  const double *q, *w, *dlnf;
  int hint[DEB_NSPLINE];
  bool lambda;  // w0 == -1 and wa == 0: dark-energy perturbations frozen
  // input tangents (gradient kernels): dcos[ndir][24], dtab[ndir][stride]
  const double *dcos;
  const double *dtab;
  int64_t stride;
  int ndir;
};

// deb_cosmo_t field indices
enum : int {
  F_GRHOM = 0, F_GRHOG, F_GRHOR, F_OMEGAM, F_OMEGAB, F_OMEGADE, F_OMEGAK, F_NEFF, F_NMNU, F_AMNU, F_W0, F_WA,
  F_CS2DE, F_YHE, F_H0, F_TAUMIN
};
constexpr int COSMO_DOUBLES = 24;

// cosmology scalar f as a T-compatible parameter: plain double, or (for dn
// types) the value with its input tangents in components 1..ndir
template <class T>
__device__ __forceinline__ ParT<T> cv(const Ctx &cx, int f) {
  const double v = reinterpret_cast<const double *>(cx.c)[f];
  if constexpr (is_dn<T>::value) {
    T r;
    r = v;
#pragma unroll
    for (int j = 0; j + 1 < T::size; ++j)
      if (j < cx.ndir) r.d[j + 1] = cx.dcos[j * COSMO_DOUBLES + f];
    return r;
  } else {
    return v;
  }
}

// spline s at x: dn types also carry the knots' input tangents (x, y and S)
template <class T>
__device__ __forceinline__ T spl_at(Ctx &cx, int s, T xv) {
  if constexpr (is_dn<T>::value) {
    const Spl &sp = cx.sp[s];
    const int i = spl_interval(sp, vval(xv), cx.hint[s]);
    auto knot = [&](int part, int idx) {
      const double *base = part == 0 ? sp.x : (part == 1 ? sp.y : sp.S);
      T r;
      r = base[idx];
#pragma unroll
      for (int j = 0; j + 1 < T::size; ++j)
        if (j < cx.ndir) r.d[j + 1] = cx.dtab[j * cx.stride + sp.off + part * sp.n + idx];
      return r;
    };
    T x0 = knot(0, i), x1 = knot(0, i + 1);
    T h = x1 - x0;
    T t = (xv - x0) / h;
    T A = 1.0 - t;
    T B = t;
    return A * knot(1, i) + B * knot(1, i + 1) +
           ((A * A * A - A) * knot(2, i) + (B * B * B - B) * knot(2, i + 1)) * (h * h / 6.0);
  } else {
    return spl_eval(cx.sp[s], xv, cx.hint[s]);
  }
}

// rho_Q(a) / rho_Q(1) = a^{-3(1+w0+wa)} exp(3 (a-1) wa); for dn types the
// exponent's own tangent enters through exp((e - e0) log a)
// (one exponential of -3 (1 + w0 + wa) log a + 3 (a - 1) wa; the exponent
// carries the parameters' tangents for dn types)
template <class T>
__device__ __forceinline__ T rho_de(T a, T loga, ParT<T> w0, ParT<T> wa) {
  return dexp((-3.0 * (1.0 + w0 + wa)) * loga + 3.0 * (a - 1.0) * wa);
}

// 1/sqrt(x): refined hardware estimate for plain doubles
template <class T>
__device__ __forceinline__ T rsqrt_t(T x) {
  if constexpr (std::is_same<T, double>::value) return rsq_nr(x);
  else return 1.0 / dsqrt(x);
}

// 1/x: refined hardware estimate for plain doubles
template <class T>
__device__ __forceinline__ T rcp_t(T x) {
  if constexpr (std::is_same<T, double>::value) return rcp_nr(x);
  else return 1.0 / x;
}

// background quantities at a, with the reciprocals 1/a, 1/a^2 and 1/(aH) that
// the row coefficients use (taken once per evaluation, not per row)
template <typename T>
struct Bg {
  T a, aH, opac, cs2, pb43, rhoQ, w, ca2;
  T ia, ia2, iaH;
};



// background at scale factor a (get_aprimeoa background.py:100-122 and the
// thermodynamics lookups of perturbations.py:176-218)
template <typename T>
__device__ __forceinline__ Bg<T> background(Ctx &cx, T a) {
  using P = ParT<T>;
  const P grhom = cv<T>(cx, F_GRHOM), grhog = cv<T>(cx, F_GRHOG), grhor = cv<T>(cx, F_GRHOR);
  const P Omegam = cv<T>(cx, F_OMEGAM), Omegab = cv<T>(cx, F_OMEGAB), OmegaDE = cv<T>(cx, F_OMEGADE);
  const P Omegak = cv<T>(cx, F_OMEGAK), Neff = cv<T>(cx, F_NEFF), Nmnu = cv<T>(cx, F_NMNU);
  const P w0 = cv<T>(cx, F_W0), wa = cv<T>(cx, F_WA), YHe = cv<T>(cx, F_YHE), H0 = cv<T>(cx, F_H0);
  Bg<T> b;
  b.a = a;
  T loga = dlog(a);
  T cs2a, xe, lrhonu;
  if constexpr (is_dn<T>::value) {
    cs2a = spl_at<T>(cx, DEB_SPL_CS2A_LOGA, loga);
    xe = spl_at<T>(cx, DEB_SPL_XE_LOGA, loga);
    lrhonu = spl_at<T>(cx, DEB_SPL_LOGRHONU_LOGA, loga);
  } else {
    const Spl sp3[3] = {cx.sp[DEB_SPL_CS2A_LOGA], cx.sp[DEB_SPL_XE_LOGA], cx.sp[DEB_SPL_LOGRHONU_LOGA]};
    int *const h3[3] = {&cx.hint[DEB_SPL_CS2A_LOGA], &cx.hint[DEB_SPL_XE_LOGA], &cx.hint[DEB_SPL_LOGRHONU_LOGA]};
    T r3[3];
    spl_eval3<T>(sp3, loga, h3, r3);
    cs2a = r3[0];
    xe = r3[1];
    lrhonu = r3[2];
  }
  b.ia = 1.0 / a;
  b.ia2 = b.ia * b.ia;
  b.cs2 = cs2a * b.ia;
  T rhonu = dexp(lrhonu);
  b.pb43 = (4.0 / 3.0) * (grhog / (grhom * Omegab)) * b.ia;
  b.w = w0 + wa * (1.0 - a);
  b.rhoQ = rho_de<T>(a, loga, w0, wa);
  T a2 = a * a;
  T grho = grhom * Omegam * b.ia + (grhog + grhor * (Neff + Nmnu * rhonu)) * b.ia2 + grhom * OmegaDE * b.rhoQ * a2 +
           grhom * Omegak;
  b.aH = dsqrt(grho * (1.0 / 3.0));
  b.iaH = 1.0 / b.aH;
  T wprime = -wa * b.aH * a;
  b.ca2 = b.w - wprime * (1.0 / 3.0) / ((1.0 + b.w) + 1e-6) * b.iaH;
  const P akthom = 2.3038921003709498e-9 * (1.0 - YHe) * Omegab * H0 * H0;
  b.opac = xe * akthom * b.ia2;
  return b;
}


template <typename T>
struct Coef {
  T sub, diag, sup;   // local tridiagonal part of J
  T uh, ueta, upi;    // where h', eta', Pi enter the row
  T ch, ceta, cpi;    // contributions of this variable to h', eta', Pi
  T c1;               // contribution to f_1 = -(dgrho + 3 dgpres) a
  T leaf;             // coupling to the leaf partner (delta_gamma <-> theta_gamma)
};

// coefficient fields of a row
enum : int { C_SUB = 0, C_DIAG, C_SUP, C_UH, C_UETA, C_UPI, C_CH, C_CETA, C_CPI, C_C1, C_LEAF };

// The coefficient fields of one row (model_synchronous, perturbations.py:
// 84-371), each passed to sink(field, value): the equations as they are
// written, one case per row type, each case setting each of its fields once.
// No kernel runs this form or row_coef_wave below; it is what the host
// emulation checks the kernels' form (row_consts, row_lin) against, row by row.
template <typename T, class Sink>
__device__ __forceinline__ void row_visit(uint32_t d, const Bg<T> &b, const Ctx &cx, double invtau, Sink sink) {
  using P = ParT<T>;
  const P grhom = cv<T>(cx, F_GRHOM), grhog = cv<T>(cx, F_GRHOG), grhor = cv<T>(cx, F_GRHOR);
  const P Omegam = cv<T>(cx, F_OMEGAM), Omegab = cv<T>(cx, F_OMEGAB), OmegaDE = cv<T>(cx, F_OMEGADE);
  const P Neff = cv<T>(cx, F_NEFF), Nmnu = cv<T>(cx, F_NMNU), cs2DE = cv<T>(cx, F_CS2DE);
  const double k = cx.k, k2 = k * k;
  const double ik2 = 1.0 / k2, hk2 = 0.5 * ik2;  // wave-uniform
  const uint32_t t = rd_type(d);
  const double l = (double)rd_l(d);
  const int qi = (int)rd_q(d);
  const T a = b.a;
  const T ia = b.ia, ia2 = b.ia2, iaH = b.iaH;
  const P Omegac = Omegam - Omegab;
  // multipole couplings l/(2l+1) and (l+1)/(2l+1), and the massive-nu velocity
  // of the row's momentum bin: evaluated once here rather than in each of the
  // (divergent) row cases that use them
  const double il = rcp_nr(2.0 * l + 1.0);
  const double lsub = l * il, lsup = (l + 1.0) * il;
  const bool qrow = t >= R_Q0 && t <= R_QLMAX;
  T vq = tconst<T>(1.0), ivq = tconst<T>(1.0);  // v_q and 1/v_q = sqrt(1 + x^2)
  if (qrow) {
    const T aq = a * (cv<T>(cx, F_AMNU) * rcp_nr(cx.q[qi]));
    const T s2 = 1.0 + aq * aq;
    vq = rsqrt_t<T>(s2);
    ivq = s2 * vq;
  }
  switch (t) {
    case R_ETA:
      sink(std::integral_constant<int, C_UETA>{}, 1.0);
      sink(std::integral_constant<int, C_CH>{}, (2.0 * k2) * iaH);
      break;
    case R_DC: {
      const P rc = grhom * Omegac;
      sink(std::integral_constant<int, C_SUP>{}, -1.0);
      sink(std::integral_constant<int, C_UH>{}, -0.5);
      sink(std::integral_constant<int, C_CH>{}, rc * ia * iaH);
      sink(std::integral_constant<int, C_C1>{}, -rc);
      break;
    }
    case R_TC:
      sink(std::integral_constant<int, C_DIAG>{}, -b.aH);
      sink(std::integral_constant<int, C_CETA>{}, grhom * Omegac * ia * hk2);
      break;
    case R_DB: {
      const P rb = grhom * Omegab;
      sink(std::integral_constant<int, C_SUP>{}, -1.0);
      sink(std::integral_constant<int, C_UH>{}, -0.5);
      sink(std::integral_constant<int, C_CH>{}, rb * ia * iaH);
      sink(std::integral_constant<int, C_C1>{}, -rb);
      break;
    }
    case R_TB: {
      const T po = b.pb43 * b.opac;
      sink(std::integral_constant<int, C_SUB>{}, k2 * b.cs2);
      sink(std::integral_constant<int, C_DIAG>{}, -b.aH - po);
      sink(std::integral_constant<int, C_SUP>{}, po);
      sink(std::integral_constant<int, C_CETA>{}, grhom * Omegab * ia * hk2);
      break;
    }
    case R_DG:
      sink(std::integral_constant<int, C_LEAF>{}, -4.0 / 3.0);
      sink(std::integral_constant<int, C_UH>{}, -2.0 / 3.0);
      sink(std::integral_constant<int, C_CH>{}, grhog * ia2 * iaH);
      sink(std::integral_constant<int, C_C1>{}, (-2.0 * grhog) * ia);
      break;
    case R_TG:
      sink(std::integral_constant<int, C_SUB>{}, b.opac);
      sink(std::integral_constant<int, C_DIAG>{}, -b.opac);
      sink(std::integral_constant<int, C_SUP>{}, -0.5 * k2);
      sink(std::integral_constant<int, C_LEAF>{}, 0.25 * k2);
      sink(std::integral_constant<int, C_CETA>{}, (4.0 / 3.0) * grhog * ia2 * hk2);
      break;
    case R_F2:
      sink(std::integral_constant<int, C_SUB>{}, 8.0 / 15.0);
      sink(std::integral_constant<int, C_DIAG>{}, -b.opac);
      sink(std::integral_constant<int, C_SUP>{}, -0.6 * k);
      sink(std::integral_constant<int, C_UH>{}, 4.0 / 15.0);
      sink(std::integral_constant<int, C_UETA>{}, 8.0 / 5.0);
      sink(std::integral_constant<int, C_UPI>{}, 0.1 * b.opac);
      sink(std::integral_constant<int, C_CPI>{}, 1.0);
      break;
    case R_FL:
      sink(std::integral_constant<int, C_SUB>{}, k * lsub);
      sink(std::integral_constant<int, C_DIAG>{}, -b.opac);
      sink(std::integral_constant<int, C_SUP>{}, -k * lsup);
      break;
    case R_FLMAX:
      sink(std::integral_constant<int, C_SUB>{}, k);
      sink(std::integral_constant<int, C_DIAG>{}, -(l + 1.0) * invtau - b.opac);
      break;
    case R_G0:
      sink(std::integral_constant<int, C_DIAG>{}, -b.opac);
      sink(std::integral_constant<int, C_SUP>{}, -k);
      sink(std::integral_constant<int, C_UPI>{}, 0.5 * b.opac);
      sink(std::integral_constant<int, C_CPI>{}, 1.0);
      break;
    case R_GL:
      sink(std::integral_constant<int, C_SUB>{}, k * lsub);
      sink(std::integral_constant<int, C_DIAG>{}, -b.opac);
      sink(std::integral_constant<int, C_SUP>{}, -k * lsup);
      break;
    case R_G2:
      sink(std::integral_constant<int, C_SUB>{}, 0.4 * k);
      sink(std::integral_constant<int, C_DIAG>{}, -b.opac);
      sink(std::integral_constant<int, C_SUP>{}, -0.6 * k);
      sink(std::integral_constant<int, C_UPI>{}, 0.1 * b.opac);
      sink(std::integral_constant<int, C_CPI>{}, 1.0);
      break;
    case R_GLMAX:
      sink(std::integral_constant<int, C_SUB>{}, k);
      sink(std::integral_constant<int, C_DIAG>{}, -(l + 1.0) * invtau - b.opac);
      break;
    case R_DR: {
      const P rr = grhor * Neff;
      sink(std::integral_constant<int, C_SUP>{}, -4.0 / 3.0);
      sink(std::integral_constant<int, C_UH>{}, -2.0 / 3.0);
      sink(std::integral_constant<int, C_CH>{}, rr * ia2 * iaH);
      sink(std::integral_constant<int, C_C1>{}, (-2.0 * rr) * ia);
      break;
    }
    case R_TR:
      sink(std::integral_constant<int, C_SUB>{}, 0.25 * k2);
      sink(std::integral_constant<int, C_SUP>{}, -0.5 * k2);
      sink(std::integral_constant<int, C_CETA>{}, (4.0 / 3.0) * Neff * grhor * ia2 * hk2);
      break;
    case R_FR2:
      sink(std::integral_constant<int, C_SUB>{}, 8.0 / 15.0);
      sink(std::integral_constant<int, C_SUP>{}, -0.6 * k);
      sink(std::integral_constant<int, C_UH>{}, 4.0 / 15.0);
      sink(std::integral_constant<int, C_UETA>{}, 8.0 / 5.0);
      break;
    case R_FRL:
      sink(std::integral_constant<int, C_SUB>{}, k * lsub);
      sink(std::integral_constant<int, C_SUP>{}, -k * lsup);
      break;
    case R_FRLMAX:
      sink(std::integral_constant<int, C_SUB>{}, k);
      sink(std::integral_constant<int, C_DIAG>{}, -(l + 1.0) * invtau);
      break;
    case R_Q0: {
      const P rn = grhor * Nmnu * cx.w[qi];
      sink(std::integral_constant<int, C_SUP>{}, -k * vq);
      sink(std::integral_constant<int, C_UH>{}, cx.dlnf[qi] * (1.0 / 6.0));
      sink(std::integral_constant<int, C_CH>{}, rn * ivq * ia2 * iaH);
      sink(std::integral_constant<int, C_C1>{}, -(rn * (ivq + vq)) * ia);
      break;
    }
    case R_Q1: {
      const T kv = k * vq;
      sink(std::integral_constant<int, C_SUB>{}, kv * (1.0 / 3.0));
      sink(std::integral_constant<int, C_SUP>{}, kv * (-2.0 / 3.0));
      sink(std::integral_constant<int, C_CETA>{}, Nmnu * grhor * k * cx.w[qi] * ia2 * hk2);
      break;
    }
    case R_Q2: {
      const T kv = k * vq;
      sink(std::integral_constant<int, C_SUB>{}, 0.4 * kv);
      sink(std::integral_constant<int, C_SUP>{}, -0.6 * kv);
      sink(std::integral_constant<int, C_UH>{}, cx.dlnf[qi] * (-1.0 / 15.0));
      sink(std::integral_constant<int, C_UETA>{}, -0.4 * cx.dlnf[qi]);
      break;
    }
    case R_QL: {
      const T kv = k * vq;
      sink(std::integral_constant<int, C_SUB>{}, kv * lsub);
      sink(std::integral_constant<int, C_SUP>{}, -kv * lsup);
      break;
    }
    case R_QLMAX: {
      sink(std::integral_constant<int, C_SUB>{}, k * vq);
      sink(std::integral_constant<int, C_DIAG>{}, -(l + 1.0) * invtau);
      break;
    }
    case R_DQ:
      if (!cx.lambda) {
        const P cs2Q = cs2DE;
        T opw = 1.0 + b.w;
        sink(std::integral_constant<int, C_DIAG>{}, -3.0 * (cs2Q - b.w) * b.aH);
        sink(std::integral_constant<int, C_SUP>{}, -opw - 9.0 * opw * (cs2Q - b.ca2) * b.aH * b.aH * ik2);
        sink(std::integral_constant<int, C_UH>{}, -0.5 * opw);
        T rq = grhom * OmegaDE * b.rhoQ * (a * a);
        sink(std::integral_constant<int, C_CH>{}, rq * iaH);
        sink(std::integral_constant<int, C_C1>{}, -a * (rq + 3.0 * cs2Q * rq));
      }
      break;
    case R_TQ:
      if (!cx.lambda) {
        const P cs2Q = cs2DE;
        T opw = 1.0 + b.w;
        sink(std::integral_constant<int, C_SUB>{}, cs2Q / opw * k2);
        sink(std::integral_constant<int, C_DIAG>{}, -(1.0 - 3.0 * cs2Q) * b.aH);
        T rq = grhom * OmegaDE * b.rhoQ * (a * a);
        sink(std::integral_constant<int, C_CETA>{}, opw * rq * hk2);
        sink(std::integral_constant<int, C_C1>{}, -a * (3.0 * (cs2Q - b.ca2) * (3.0 * b.aH * ik2) * opw * rq));
      }
      break;
    default:
      break;
  }
}


// all coefficients of a row (fields not set by the row are zero)
template <typename T>
__device__ __forceinline__ Coef<T> row_coef(uint32_t d, const Bg<T> &b, const Ctx &cx, double invtau) {
  T v[11];
#pragma unroll
  for (int i = 0; i < 11; ++i) v[i] = 0.0;
  // (accumulating rather than assigning keeps the compiler from merging the
  // cases' stores into one store at a variable index, which would move v to
  // the stack)
  row_visit<T>(d, b, cx, invtau, [&](auto f, const auto &x) __attribute__((always_inline)) {
    v[decltype(f)::value] = v[decltype(f)::value] + x;
  });
  Coef<T> r;
  r.sub = v[C_SUB]; r.diag = v[C_DIAG]; r.sup = v[C_SUP];
  r.uh = v[C_UH]; r.ueta = v[C_UETA]; r.upi = v[C_UPI];
  r.ch = v[C_CH]; r.ceta = v[C_CETA]; r.cpi = v[C_CPI]; r.c1 = v[C_C1]; r.leaf = v[C_LEAF];
  return r;
}

// row_coef organised for the wave instead of as a divergent switch, with the
// same formulas in the same operation order (the host emulation compares the
// two; no kernel runs it): the chain rows (hierarchies, any slot) by per-lane
// selects among their formulas; with slot0, the fixed-lane rows of slot 0 as
// wave-uniform values selected by lane.
template <typename T>
__device__ __forceinline__ Coef<T> row_coef_wave(uint32_t d, const Bg<T> &b, const Ctx &cx, double invtau,
                                                 bool slot0) {
  using P = ParT<T>;
  const T zero = tconst<T>(0.0);
  auto c = [](double v) { return tconst<T>(v); };
  const P grhom = cv<T>(cx, F_GRHOM), grhog = cv<T>(cx, F_GRHOG), grhor = cv<T>(cx, F_GRHOR);
  const P Neff = cv<T>(cx, F_NEFF), Nmnu = cv<T>(cx, F_NMNU);
  const double k = cx.k, k2 = k * k;
  const double ik2 = 1.0 / k2, hk2 = 0.5 * ik2;
  const uint32_t t = rd_type(d);
  const double l = (double)rd_l(d);
  const bool F2 = t == R_F2, FL = t == R_FL, FLM = t == R_FLMAX, G0 = t == R_G0, GL = t == R_GL, G2 = t == R_G2,
             GLM = t == R_GLMAX, DR = t == R_DR, TR = t == R_TR, FR2 = t == R_FR2, FRL = t == R_FRL,
             FRLM = t == R_FRLMAX, Q0 = t == R_Q0, Q1 = t == R_Q1, Q2 = t == R_Q2, QL = t == R_QL,
             QLM = t == R_QLMAX;
  const bool qrow = t >= R_Q0 && t <= R_QLMAX;
  const int qi = qrow ? (int)rd_q(d) : 0;
  const T ia = b.ia, ia2 = b.ia2, iaH = b.iaH;
  const double il = rcp_nr(2.0 * l + 1.0);
  const double lsub = l * il, lsup = (l + 1.0) * il;
  // v_q and 1/v_q of the row's bin (1 on other rows); k v_q multiplies the
  // couplings of every chain (k v_q = k exactly where v_q = 1)
  T vq = c(1.0), ivq = c(1.0);
  {
    const T aq = b.a * (cv<T>(cx, F_AMNU) * rcp_nr(cx.q[qi]));
    const T s2 = 1.0 + aq * aq;
    const T v = rsqrt_t<T>(s2);
    vq = qrow ? v : c(1.0);
    ivq = qrow ? s2 * v : c(1.0);
  }
  const T kv = k * vq;
  const double wq = cx.w[qi], dl = cx.dlnf[qi];
  Coef<T> r;
  // sub-diagonal
  double cs = 0.0;
  cs = (FL || GL || FRL || QL) ? lsub : cs;
  cs = (FLM || GLM || FRLM || QLM) ? 1.0 : cs;
  cs = (G2 || Q2) ? 0.4 : cs;
  cs = Q1 ? 1.0 / 3.0 : cs;
  r.sub = kv * cs;
  r.sub = (F2 || FR2) ? c(8.0 / 15.0) : r.sub;
  r.sub = TR ? c(0.25 * k2) : r.sub;
  // diagonal: opacity of the photon rows, free streaming out of the last multipole
  const bool photon = F2 || FL || FLM || G0 || GL || G2 || GLM;
  r.diag = photon ? -b.opac : zero;
  r.diag = (FLM || GLM) ? -(l + 1.0) * invtau - b.opac : r.diag;
  r.diag = (FRLM || QLM) ? c(-(l + 1.0) * invtau) : r.diag;
  // super-diagonal
  double cp = 0.0;
  cp = (F2 || G2 || FR2 || Q2) ? 0.6 : cp;
  cp = (FL || GL || FRL || QL) ? lsup : cp;
  cp = (G0 || Q0) ? 1.0 : cp;
  cp = Q1 ? 2.0 / 3.0 : cp;
  r.sup = cp != 0.0 ? -(kv * cp) : zero;
  r.sup = DR ? c(-4.0 / 3.0) : r.sup;
  r.sup = TR ? c(-0.5 * k2) : r.sup;
  // where h', eta', Pi enter
  r.uh = (F2 || FR2) ? c(4.0 / 15.0) : zero;
  r.uh = DR ? c(-2.0 / 3.0) : r.uh;
  r.uh = Q0 ? c(dl * (1.0 / 6.0)) : r.uh;
  r.uh = Q2 ? c(dl * (-1.0 / 15.0)) : r.uh;
  r.ueta = (F2 || FR2) ? c(8.0 / 5.0) : (Q2 ? c(-0.4 * dl) : zero);
  r.upi = (F2 || G2) ? 0.1 * b.opac : (G0 ? 0.5 * b.opac : zero);
  // contributions to h', eta', Pi and f_1
  const P rr = grhor * Neff;
  const P rn = grhor * Nmnu * wq;
  r.ch = DR ? rr * ia2 * iaH : (Q0 ? rn * ivq * ia2 * iaH : zero);
  r.ceta = TR ? (4.0 / 3.0) * Neff * grhor * ia2 * hk2 : (Q1 ? Nmnu * grhor * k * wq * ia2 * hk2 : zero);
  r.cpi = (F2 || G0 || G2) ? c(1.0) : zero;
  r.c1 = DR ? (-2.0 * rr) * ia : (Q0 ? -(rn * (ivq + vq)) * ia : zero);
  r.leaf = zero;
  if (slot0) {
    const int lane = lane_id();
    const P Omegam = cv<T>(cx, F_OMEGAM), Omegab = cv<T>(cx, F_OMEGAB);
    const P Omegac = Omegam - Omegab;
    const T a = b.a;
    // eta
    r.ueta = lane == L_ETA ? c(1.0) : r.ueta;
    r.ch = lane == L_ETA ? (2.0 * k2) * iaH : r.ch;
    // delta_c, delta_b
    const P rc = grhom * Omegac, rb = grhom * Omegab;
    const bool dcb = lane == L_DC || lane == L_DB;
    const P rcb = lane == L_DC ? rc : rb;
    r.sup = dcb ? c(-1.0) : r.sup;
    r.uh = dcb ? c(-0.5) : r.uh;
    r.ch = dcb ? rcb * ia * iaH : r.ch;
    r.c1 = dcb ? zero - rcb : r.c1;
    // theta_c
    r.diag = lane == L_TC ? -b.aH : r.diag;
    r.ceta = lane == L_TC ? grhom * Omegac * ia * hk2 : r.ceta;
    // theta_b
    {
      const T po = b.pb43 * b.opac;
      const bool on = lane == L_TB;
      r.sub = on ? k2 * b.cs2 : r.sub;
      r.diag = on ? -b.aH - po : r.diag;
      r.sup = on ? po : r.sup;
      r.ceta = on ? grhom * Omegab * ia * hk2 : r.ceta;
    }
    // delta_gamma
    {
      const bool on = lane == L_DG;
      r.leaf = on ? c(-4.0 / 3.0) : r.leaf;
      r.uh = on ? c(-2.0 / 3.0) : r.uh;
      r.ch = on ? grhog * ia2 * iaH : r.ch;
      r.c1 = on ? (-2.0 * grhog) * ia : r.c1;
    }
    // theta_gamma
    {
      const bool on = lane == L_TG;
      r.sub = on ? b.opac : r.sub;
      r.diag = on ? -b.opac : r.diag;
      r.sup = on ? c(-0.5 * k2) : r.sup;
      r.leaf = on ? c(0.25 * k2) : r.leaf;
      r.ceta = on ? (4.0 / 3.0) * grhog * ia2 * hk2 : r.ceta;
    }
    // dark-energy fluid (frozen for a cosmological constant)
    if (!cx.lambda) {
      const P OmegaDE = cv<T>(cx, F_OMEGADE), cs2Q = cv<T>(cx, F_CS2DE);
      const T opw = 1.0 + b.w;
      const T rq = grhom * OmegaDE * b.rhoQ * (a * a);
      const bool dq = lane == L_DQ, tq = lane == L_TQ;
      r.diag = dq ? -3.0 * (cs2Q - b.w) * b.aH : r.diag;
      r.sup = dq ? -opw - 9.0 * opw * (cs2Q - b.ca2) * b.aH * b.aH * ik2 : r.sup;
      r.uh = dq ? -0.5 * opw : r.uh;
      r.ch = dq ? rq * iaH : r.ch;
      r.c1 = dq ? -a * (rq + 3.0 * cs2Q * rq) : r.c1;
      r.sub = tq ? cs2Q / opw * k2 : r.sub;
      r.diag = tq ? -(1.0 - 3.0 * cs2Q) * b.aH : r.diag;
      r.ceta = tq ? opw * rq * hk2 : r.ceta;
      r.c1 = tq ? -a * (3.0 * (cs2Q - b.ca2) * (3.0 * b.aH * ik2) * opw * rq) : r.c1;
    }
  }
  return r;
}

// ---------------------------------------------------------------------------
// The rows as constants times background features.  Along one mode every
// coefficient of a row is a number that depends on the row, k and the
// cosmology only, times one of a few wave-uniform functions of a (the opacity,
// aH, 1/a, ...) and, on massive-nu rows, the bin velocity: the numbers are
// formed once per mode (row_consts) and a right-hand side costs about a dozen
// multiplications per slot, where the selects of row_coef_wave took about two
// hundred instructions.  The same products as row_visit up to the order of the
// factors (within 2 units of 2^-52 of it on every row).
template <int NS>
struct RowK {
  double sub[NS], sup[NS];             // neighbours (times v_q on massive-nu rows)
  double ph[NS];                       // 1 on photon rows (-opac on the diagonal)
  double tr[NS];                       // l + 1 on truncation rows, else 0
  double uh[NS], ueta[NS], upi[NS];    // where h', eta', Pi enter (upi times opac)
  double ch[NS], ceta[NS], cpi[NS];    // contributions to h', eta', Pi
  double aq[NS];                       // m_nu / q on massive-nu rows, else 0
  double nd[NS], ne[NS];               // neutrino rows: weight of the density in ch and c1, in ceta
  double leaf, dah;                    // slot 0: leaf coupling, -aH on the diagonal
  uint32_t qmask;                      // slots that hold massive-nu rows (wave-uniform)
};

template <int NS>
__device__ __forceinline__ void row_consts(const uint32_t (&rd)[NS], const Ctx &cx, RowK<NS> &K) {
  const int lane = lane_id();
  const deb_cosmo_t &c = *cx.c;
  const double k = cx.k, k2 = k * k, hk2 = 0.5 / k2;
  K.qmask = 0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const uint32_t t = rd_type(rd[s]);
    const double l = (double)rd_l(rd[s]);
    const bool F2 = t == R_F2, FL = t == R_FL, FLM = t == R_FLMAX, G0 = t == R_G0, GL = t == R_GL, G2 = t == R_G2,
               GLM = t == R_GLMAX, DR = t == R_DR, TR = t == R_TR, FR2 = t == R_FR2, FRL = t == R_FRL,
               FRLM = t == R_FRLMAX, Q0 = t == R_Q0, Q1 = t == R_Q1, Q2 = t == R_Q2, QL = t == R_QL,
               QLM = t == R_QLMAX;
    const bool qrow = t >= R_Q0 && t <= R_QLMAX;
    const int qi = qrow ? (int)rd_q(rd[s]) : 0;
    const double wq = cx.w[qi], dl = cx.dlnf[qi];
    const double il = rcp_nr(2.0 * l + 1.0);
    const bool mid = FL || GL || FRL || QL, last = FLM || GLM || FRLM || QLM;
    double v = 0.0;
    v = mid ? k * (l * il) : v;
    v = last ? k : v;
    v = (G2 || Q2) ? 0.4 * k : v;
    v = Q1 ? k * (1.0 / 3.0) : v;
    v = (F2 || FR2) ? 8.0 / 15.0 : v;
    K.sub[s] = TR ? 0.25 * k2 : v;
    v = 0.0;
    v = (F2 || G2 || FR2 || Q2) ? -(0.6 * k) : v;
    v = mid ? -(k * ((l + 1.0) * il)) : v;
    v = (G0 || Q0) ? -k : v;
    v = Q1 ? -(k * (2.0 / 3.0)) : v;
    v = DR ? -4.0 / 3.0 : v;
    K.sup[s] = TR ? -0.5 * k2 : v;
    K.ph[s] = (F2 || FL || FLM || G0 || GL || G2 || GLM) ? 1.0 : 0.0;
    K.tr[s] = last ? l + 1.0 : 0.0;
    v = (F2 || FR2) ? 4.0 / 15.0 : 0.0;
    v = DR ? -2.0 / 3.0 : v;
    v = Q0 ? dl * (1.0 / 6.0) : v;
    K.uh[s] = Q2 ? dl * (-1.0 / 15.0) : v;
    K.ueta[s] = (F2 || FR2) ? 8.0 / 5.0 : (Q2 ? -0.4 * dl : 0.0);
    K.upi[s] = (F2 || G2) ? 0.1 : (G0 ? 0.5 : 0.0);
    K.ch[s] = DR ? c.grhor * c.Neff : (Q0 ? c.grhor * c.Nmnu * wq : 0.0);
    K.ceta[s] = TR ? (4.0 / 3.0) * c.Neff * c.grhor * hk2 : (Q1 ? c.Nmnu * c.grhor * k * wq * hk2 : 0.0);
    K.cpi[s] = (F2 || G0 || G2) ? 1.0 : 0.0;
    K.aq[s] = qrow ? c.amnu * rcp_nr(cx.q[qi]) : 0.0;
    K.nd[s] = DR ? 1.0 : (Q0 ? wq : 0.0);
    K.ne[s] = TR ? (4.0 / 3.0) * hk2 : (Q1 ? k * wq * hk2 : 0.0);
    if (__ballot(qrow) != 0) K.qmask |= 1u << s;
    if (s == 0) {
      const double rc = c.grhom * (c.Omegam - c.Omegab), rb = c.grhom * c.Omegab;
      const bool DC = lane == L_DC, DB = lane == L_DB, TC = lane == L_TC, TB = lane == L_TB, DG = lane == L_DG,
                 TG = lane == L_TG, ETA = lane == L_ETA;
      K.sup[0] = (DC || DB) ? -1.0 : (TG ? -0.5 * k2 : K.sup[0]);
      K.ph[0] = TG ? 1.0 : K.ph[0];
      K.uh[0] = (DC || DB) ? -0.5 : (DG ? -2.0 / 3.0 : K.uh[0]);
      K.ueta[0] = ETA ? 1.0 : K.ueta[0];
      v = ETA ? 2.0 * k2 : K.ch[0];
      v = DC ? rc : v;
      v = DB ? rb : v;
      K.ch[0] = DG ? c.grhog : v;
      v = TC ? rc * hk2 : K.ceta[0];
      v = TB ? rb * hk2 : v;
      K.ceta[0] = TG ? (4.0 / 3.0) * c.grhog * hk2 : v;
      K.leaf = DG ? -4.0 / 3.0 : (TG ? 0.25 * k2 : 0.0);
      v = (TC || TB) ? 1.0 : 0.0;
      K.dah = (lane == L_TQ && !cx.lambda) ? 1.0 - 3.0 * c.cs2_DE : v;
    }
  }
}

// 1/x and component-wise selection in plain doubles and along a
__device__ __forceinline__ double rcp_a(double x) { return rcp_nr(x); }
__device__ __forceinline__ dual rcp_a(dual x) {
  const double r = rcp_nr(x.v);
  return {r, -(r * r) * x.d};
}
__device__ __forceinline__ double sel(bool c, double x, double y) { return c ? x : y; }
__device__ __forceinline__ dual sel(bool c, dual x, dual y) { return {c ? x.v : y.v, c ? x.d : y.d}; }

// log x for positive normal x, NaN otherwise: x = m 2^e with m in
// [1/sqrt 2, sqrt 2], log m = 2 atanh z, z = (m - 1) / (m + 1), |z| < 0.172,
// by its series up to z^23 (remainder below 1e-19).  Two fifths of the
// instructions of the library's log.  Within 1.02 ulp of log x (the library's
// log 0.64); opacity, sound speed, rho_Q and aH have the same error against 113
// bits with either: they are bound by the rounding of log a itself and of the
// spline's sums.
__device__ __forceinline__ double log_pos(double x) {
  const int hi = __double2hiint(x);
  int e = (hi >> 20) - 1023;
  double m = __hiloint2double((hi & 0xfffff) | 0x3ff00000, __double2loint(x));
  const bool up = m > 1.4142135623730951;
  m = up ? 0.5 * m : m;
  e = up ? e + 1 : e;
  // (the quotient corrected by its residual, the rounding of m + 1 included)
  const double f = m - 1.0, d1 = m + 1.0, rd = rcp_nr(d1), z0 = f * rd;
  const double z = fma(fma(-z0, d1, f) - z0 * (m - (d1 - 1.0)), rd, z0), w = z * z;
  double p = 2.0 / 23.0;
  p = fma(p, w, 2.0 / 21.0);
  p = fma(p, w, 2.0 / 19.0);
  p = fma(p, w, 2.0 / 17.0);
  p = fma(p, w, 2.0 / 15.0);
  p = fma(p, w, 2.0 / 13.0);
  p = fma(p, w, 2.0 / 11.0);
  p = fma(p, w, 2.0 / 9.0);
  p = fma(p, w, 2.0 / 7.0);
  p = fma(p, w, 2.0 / 5.0);
  p = fma(p, w, 2.0 / 3.0);
  const double d = (double)e;
  // ln 2 in the two parts that fdlibm publishes, the first exact in products with e
  const double r = fma(d, 6.93147180369123816490e-01, fma(2.0, z, fma(z * w, p, d * 1.90821492927058770002e-10)));
  return x >= 2.2250738585072014e-308 && x <= 1.7976931348623157e308 ? r : __builtin_nan("");
}

// ---------------------------------------------------------------------------
// The background of one mode's right-hand sides.  The cosmology's numbers are
// combined once per mode.  The three splines' knots live in registers, one
// interval per lane: lane 4 w + j holds interval base_j + w of spline j, so
// sixteen consecutive intervals of each are at hand, a ballot finds the lanes
// whose interval holds log a, and memory is read only when log a leaves a
// window (from six knots per right-hand side through the caches before).  With
// the launch constants kept uniform (deb_kargs.h): 64 cosmologies x 256 k at lmax
// 32 227 -> 165 ms, one step of 1500 states 138 -> 94.7 us.
struct BgCache {
  const double *x;  // the lane's spline: knots x, then y, then S, n each
  int n;
  double xlo, xhi;  // the lane's interval, the first and the last one open to infinity
  double x0, ih, y0, y1, s0, s1;  // its knots: 1/h, S h^2 / 6
  double gm, ggr, gn, gde, gk;    // densities: grhom Omega_m, grhog + grhor Neff, grhor Nmnu, grhom Omega_DE, grhom Omega_k
  double w0, wa, e1;              // e1 = -3 (1 + w0 + wa)
  double kth, pb;                 // opacity / x_e a^2; (4/3) rho_g / rho_b a
  double cs2Q, k2, ik2;
  bool lambda;
};

__device__ __forceinline__ void bg_set_k(BgCache &g, double k) {
  g.k2 = k * k;
  g.ik2 = 1.0 / g.k2;
}

__device__ __forceinline__ void bg_init(const Ctx &cx, BgCache &g) {
  const deb_cosmo_t &c = *cx.c;
  const int j = lane_id() & 3;
  const Spl s0 = cx.sp[DEB_SPL_CS2A_LOGA], s1 = cx.sp[DEB_SPL_XE_LOGA], s2 = cx.sp[DEB_SPL_LOGRHONU_LOGA];
  g.x = j == 0 ? s0.x : (j == 1 ? s1.x : s2.x);
  g.n = j == 0 ? s0.n : (j == 1 ? s1.n : s2.n);
  g.xlo = INFINITY;  // no interval yet
  g.xhi = g.x0 = g.ih = g.y0 = g.y1 = g.s0 = g.s1 = 0.0;
  g.gm = c.grhom * c.Omegam;
  g.ggr = c.grhog + c.grhor * c.Neff;
  g.gn = c.grhor * c.Nmnu;
  g.gde = c.grhom * c.OmegaDE;
  g.gk = c.grhom * c.Omegak;
  g.w0 = c.w_DE_0;
  g.wa = c.w_DE_a;
  g.e1 = -3.0 * (1.0 + c.w_DE_0 + c.w_DE_a);
  g.kth = 2.3038921003709498e-9 * (1.0 - c.YHe) * c.Omegab * c.H0 * c.H0;
  g.pb = (4.0 / 3.0) * (c.grhog / (c.grhom * c.Omegab));
  g.cs2Q = c.cs2_DE;
  g.lambda = cx.lambda;
  bg_set_k(g, cx.k);
}

// moves every spline's window so that it holds the interval of v (the rule of
// spl_interval), three intervals behind it and twelve ahead; returns the lane
// that holds the interval of the lane's own spline
__device__ __forceinline__ int bg_seek(BgCache &g, double v) {
  const double *x = g.x, *y = g.x + g.n, *S = y + g.n;
  int lo = 0, hi = g.n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (x[mid] < v) lo = mid + 1; else hi = mid;
  }
  int i = lo - 1;
  i = i < 0 ? 0 : (i > g.n - 2 ? g.n - 2 : i);
  const int base = i < 3 ? 0 : i - 3;
  const int own = base + (lane_id() >> 2);
  const int c = own > g.n - 2 ? g.n - 2 : own;
  const double x0 = x[c], x1 = x[c + 1], h = x1 - x0, h26 = h * h / 6.0;
  g.x0 = x0;
  g.ih = 1.0 / h;
  g.y0 = y[c];
  g.y1 = y[c + 1];
  g.s0 = S[c] * h26;
  g.s1 = S[c + 1] * h26;
  g.xlo = own > g.n - 2 ? INFINITY : (own == 0 ? -INFINITY : x0);
  g.xhi = own == g.n - 2 ? INFINITY : x1;
  return (i - base) * 4 + (lane_id() & 3);
}

// background quantities at a, as far as the rows need them
template <typename T>
struct BgRow {
  T a, aH, iaH, ia, ia2, opac, cs2, po, rhoQ;
};

// the spline's value at v in units of its interval, and along log a
__device__ __forceinline__ double bg_piece(const BgCache &g, double v) {
  const double B = (v - g.x0) * g.ih, A = 1.0 - B;
  return A * g.y0 + B * g.y1 + ((A * A * A - A) * g.s0 + (B * B * B - B) * g.s1);
}
__device__ __forceinline__ double bg_slope(const BgCache &g, double v) {
  const double B = (v - g.x0) * g.ih, A = 1.0 - B;
  return (g.y1 - g.y0 + ((3.0 * B * B - 1.0) * g.s1 - (3.0 * A * A - 1.0) * g.s0)) * g.ih;
}

template <typename T>
__device__ __forceinline__ BgRow<T> background_row(BgCache &g, T a) {
  constexpr bool D = !std::is_same<T, double>::value;
  const int lane = lane_id();
  const double av = vval(a);
  const double loga = log_pos(av);
  const uint64_t in = __ballot(g.xlo < loga && loga <= g.xhi);
  const uint64_t m0 = in & 0x1111111111111111ull, m1 = in & 0x2222222222222222ull, m2 = in & 0x4444444444444444ull;
  int l0, l1, l2;
  if (m0 != 0 && m1 != 0 && m2 != 0) {
    l0 = __builtin_ctzll(m0);
    l1 = __builtin_ctzll(m1);
    l2 = __builtin_ctzll(m2);
  } else {
    const int l = bg_seek(g, loga);
    l0 = __builtin_amdgcn_readlane(l, 0);
    l1 = __builtin_amdgcn_readlane(l, 1);
    l2 = __builtin_amdgcn_readlane(l, 2);
  }
  const double val = bg_piece(g, loga);
  // both exponentials at once: lane 0 that of log rho_nu, the others dark energy's
  const double lrnu = readlane(val, l2);
  const double ex = exp(lane == 0 ? lrnu : g.e1 * loga + 3.0 * (av - 1.0) * g.wa);
  BgRow<T> b;
  T cs2a, xe, rhonu;
  b.a = a;
  b.ia = rcp_a(a);
  if constexpr (D) {
    const double slope = bg_slope(g, loga);
    const double ia = b.ia.v;
    const double e0 = readlane(ex, 0), e1 = readlane(ex, 1);
    cs2a = T{readlane(val, l0), readlane(slope, l0) * ia};
    xe = T{readlane(val, l1), readlane(slope, l1) * ia};
    rhonu = T{e0, e0 * (readlane(slope, l2) * ia)};
    b.rhoQ = T{e1, e1 * (g.e1 * ia + 3.0 * g.wa)};
  } else {
    cs2a = readlane(val, l0);
    xe = readlane(val, l1);
    rhonu = readlane(ex, 0);
    b.rhoQ = readlane(ex, 1);
  }
  b.ia2 = b.ia * b.ia;
  b.cs2 = cs2a * b.ia;
  b.opac = g.kth * xe * b.ia2;
  b.po = (g.pb * b.ia) * b.opac;
  const T grho3 = (g.gm * b.ia + (g.ggr + g.gn * rhonu) * b.ia2 + g.gde * b.rhoQ * (a * a) + g.gk) * (1.0 / 3.0);
  // aH = sqrt(grho3) and its reciprocal from one estimate, the root corrected by its residual
  const double r = rsq_nr(vval(grho3));
  double h = vval(grho3) * r;
  h = fma(fma(-h, h, vval(grho3)), 0.5 * r, h);
  if constexpr (D) {
    const double hd = 0.5 * grho3.d * r;
    b.aH = T{h, hd};
    b.iaH = T{r, -hd * (r * r)};
  } else {
    b.aH = h;
    b.iaH = r;
  }
  return b;
}

// v_q = (1 + x^2)^(-1/2) and 1/v_q of x = a m_nu / q
__device__ __forceinline__ void bin_velocity(double a, double aq, double &vq, double &ivq) {
  const double x = a * aq, s2 = 1.0 + x * x;
  vq = rsq_nr(s2);
  ivq = s2 * vq;
}
__device__ __forceinline__ void bin_velocity(dual a, double aq, dual &vq, dual &ivq) {
  const double x = a.v * aq, s2 = 1.0 + x * x, hd = x * (aq * a.d);
  vq.v = rsq_nr(s2);
  ivq.v = s2 * vq.v;
  ivq.d = hd * vq.v;
  vq.d = -hd * (vq.v * vq.v * vq.v);
}

// the coefficients of slot s's rows at background b, from their constants
template <int NS, typename T>
__device__ __forceinline__ Coef<T> row_lin(const RowK<NS> &K, int s, const BgRow<T> &b, const BgCache &g,
                                           double invtau) {
  Coef<T> r;
  T vq = tconst<T>(1.0), ivq = tconst<T>(1.0);
  if ((K.qmask >> s) & 1u) bin_velocity(b.a, K.aq[s], vq, ivq);
  r.sub = K.sub[s] * vq;
  r.sup = K.sup[s] * vq;
  r.diag = -(K.ph[s] * b.opac) - K.tr[s] * invtau;
  r.uh = tconst<T>(K.uh[s]);
  r.ueta = tconst<T>(K.ueta[s]);
  r.upi = K.upi[s] * b.opac;
  r.cpi = tconst<T>(K.cpi[s]);
  r.leaf = tconst<T>(0.0);
  r.ch = K.ch[s] * (ivq * (b.ia2 * b.iaH));
  r.ceta = K.ceta[s] * b.ia2;
  r.c1 = (-K.ch[s]) * ((ivq + vq) * b.ia);
  if (s == 0) {
    const int lane = lane_id();
    const bool dcb = (lane == L_DC) | (lane == L_DB), eta = lane == L_ETA, tb = lane == L_TB, tg = lane == L_TG;
    r.leaf = tconst<T>(K.leaf);
    r.diag = r.diag - K.dah * b.aH;
    r.diag = sel(tb, r.diag - b.po, r.diag);
    r.sub = sel(tb, g.k2 * b.cs2, sel(tg, b.opac, r.sub));
    r.sup = sel(tb, b.po, r.sup);
    r.ch = sel(dcb, K.ch[0] * (b.ia * b.iaH), sel(eta, K.ch[0] * b.iaH, r.ch));
    r.c1 = sel(dcb | eta, tconst<T>(eta ? 0.0 : -K.ch[0]), r.c1);
    r.ceta = sel(tb | (lane == L_TC), K.ceta[0] * b.ia, r.ceta);
    // dark-energy fluid (frozen for a cosmological constant)
    if (!g.lambda) {
      const bool dq = lane == L_DQ, tq = lane == L_TQ;
      const T w = g.w0 + g.wa * (1.0 - b.a);
      const T opw = 1.0 + w;
      const T dc = g.cs2Q - w - (g.wa * (1.0 / 3.0)) * (b.a * rcp_a(opw + 1e-6));  // c_s^2 - c_a^2
      const T rq = g.gde * b.rhoQ * (b.a * b.a);
      const T oaH = opw * b.aH * dc;
      r.diag = sel(dq, -3.0 * (g.cs2Q - w) * b.aH, r.diag);
      r.sup = sel(dq, -opw - (9.0 * g.ik2) * (oaH * b.aH), r.sup);
      r.uh = sel(dq, -0.5 * opw, r.uh);
      r.ch = sel(dq, rq * b.iaH, r.ch);
      r.sub = sel(tq, (g.cs2Q * g.k2) * rcp_a(opw), r.sub);
      r.ceta = sel(tq, (0.5 * g.ik2) * (opw * rq), r.ceta);
      const T arq = b.a * rq;
      r.c1 = sel(dq, (-(1.0 + 3.0 * g.cs2Q)) * arq, sel(tq, (-9.0 * g.ik2) * (oaH * arq), r.c1));
    }
  }
  return r;
}

}  // namespace deb

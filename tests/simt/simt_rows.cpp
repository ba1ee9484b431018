// CPU emulation harness of the right-hand side's coefficients: the form that
// the kernels run (row_consts, background_row, row_lin) against the equations
// row by row (row_coef) and the plain background (background).  Built and run
// like simt_host (64 host threads per wavefront, sanitizers).  Test
// infrastructure only.
//
//   simt_rows <in.bin> <out.bin>
//
// in.bin: written by _write of tests/test_simt_host.py, mode 0, followed by
//   int32 na; double a[na]: the scale factors in the order of evaluation, one
//   window of the splines after the other as a solve would move them
// out.bin: double worst[4]: the largest error in units of 2^-52 times its scale
//   of the rows' values (scale: the value), the rows' derivatives along a (the
//   value times its features' logarithmic derivatives), the background's values
//   and its derivatives (scales: bounds of the rounding); int32 compared fields
#include "simt_common.h"

#include "../../disco-eb_amd/csrc/deb_forward.h"

using namespace deb;

namespace {

constexpr double EPS = 2.220446049250313e-16;

struct Worst {
  double w[4] = {0.0, 0.0, 0.0, 0.0};
  int32_t n = 0;
  // error of x against ref in units of EPS * scale; equal values need no scale
  void add(int which, double x, double ref, double scale) {
    ++n;
    if (x != ref) merge(which, std::fabs(x - ref) / (EPS * scale));
  }
  // a NaN stays
  void merge(int which, double e) {
    if (w[which] == w[which] && !(e <= w[which])) w[which] = e;
  }
};

// magnitude of the terms of spline s around log a, and its interval's width
struct Piece {
  double m, h;
  Piece(const Spl &s, double la) {
    int i = (int)(std::lower_bound(s.x, s.x + s.n, la) - s.x) - 1;
    i = std::min(std::max(i, 0), s.n - 2);
    h = s.x[i + 1] - s.x[i];
    const double t = 1.0 + std::fabs((la - s.x[i]) / h);  // beyond 2 outside the knots
    m = t * t * t * (std::fabs(s.y[i]) + std::fabs(s.y[i + 1]) + h * h / 6.0 * (std::fabs(s.S[i]) + std::fabs(s.S[i + 1])));
  }
  // bounds in EPS, log a off by dla EPS: 16 roundings of the terms, and the
  // slope (at most 3 m / h) or the curvature (6 m / h^2) times the shift
  double value(double dla) const { return 16.0 * m + dla * 3.0 * m / h; }
  double slope(double dla) const { return 48.0 * m / h + dla * 6.0 * m / (h * h); }
};

template <int NS>
void compare(const Params<NS> &P, const std::vector<double> &as, double k, bool lambda, Worst &out) {
  const int lane = lane_id();
  Ctx cx;
  make_ctx<NS>(cx, P, 0, k);
  cx.lambda = lambda;
  uint32_t rd[NS];
  for (int s = 0; s < NS; ++s) rd[s] = P.rowdesc[s][lane];
  RowK<NS> K;
  row_consts<NS>(rd, cx, K);
  BgCache g, gd;  // a solve's right-hand sides and its factorisations move one window; here one each
  bg_init(cx, g);
  bg_init(cx, gd);
  for (double a : as) {
    const double invtau = 1.0 / (30.0 + 1e4 * a);
    const BgRow<double> b = background_row<double>(g, a);
    const BgRow<dual> d = background_row<dual>(gd, mkd(a, 1.0));
    const Bg<double> rb = background<double>(cx, a);
    const Bg<dual> r = background<dual>(cx, mkd(a, 1.0));
    // the background: the same spline pieces and sums in another order, at a
    // log a that may be 2 ulp off
    const double la0 = std::log(a), dla = 2.0 * std::fabs(la0);
    const Piece pc(cx.sp[DEB_SPL_CS2A_LOGA], la0), px(cx.sp[DEB_SPL_XE_LOGA], la0), pn(cx.sp[DEB_SPL_LOGRHONU_LOGA], la0);
    auto bg = [&](double x, dual xd, dual ref, double value, double slope) {
      out.add(2, x, ref.v, value);
      out.add(2, xd.v, ref.v, value);
      out.add(3, xd.d, ref.d, slope);
    };
    const double ia = 1.0 / a, vn = 16.0 + pn.value(dla), dn_ = (64.0 + 4.0 * vn + pn.slope(dla)) * ia;
    bg(b.ia, d.ia, r.ia, 16.0 * ia, 16.0 * ia * ia);
    bg(b.ia2, d.ia2, r.ia2, 16.0 * ia * ia, 32.0 * ia * ia * ia);
    bg(b.aH, d.aH, r.aH, r.aH.v * vn, r.aH.v * dn_);
    bg(b.iaH, d.iaH, r.iaH, r.iaH.v * vn, r.iaH.v * dn_);
    const double vc = pc.value(dla) * ia, dc = (2.0 * pc.value(dla) + pc.slope(dla)) * ia * ia;
    bg(b.cs2, d.cs2, r.cs2, vc, dc);
    const double kx = g.kth * ia * ia, vx = kx * px.value(dla), dx = kx * ia * (4.0 * px.value(dla) + px.slope(dla));
    bg(b.opac, d.opac, r.opac, vx, dx);
    const double pb = g.pb * ia;
    bg(b.po, d.po, r.pb43 * r.opac, 2.0 * pb * vx, 2.0 * pb * (dx + vx * ia));
    const double e1 = std::fabs(g.e1), ea = 3.0 * std::fabs(g.wa);
    const double vq = 16.0 + 4.0 * (e1 * std::fabs(la0) + ea) + e1 * dla;
    bg(b.rhoQ, d.rhoQ, r.rhoQ, r.rhoQ.v * vq, r.rhoQ.v * (vq + 16.0) * (e1 * ia + ea));
    // the rows from one background: the equations at the kernels' values
    Bg<double> eb;
    Bg<dual> ed;
    auto same = [&](auto &e, const auto &v) {
      e.a = v.a;
      e.aH = v.aH;
      e.opac = v.opac;
      e.cs2 = v.cs2;
      e.pb43 = g.pb * v.ia;
      e.rhoQ = v.rhoQ;
      e.w = g.w0 + g.wa * (1.0 - v.a);
      e.ca2 = e.w + (g.wa * (1.0 / 3.0)) * (v.a / (1.0 + e.w + 1e-6));
      e.ia = v.ia;
      e.ia2 = v.ia2;
      e.iaH = v.iaH;
    };
    same(eb, b);
    same(ed, d);
    const double opw = 1.0 + eb.w, dw = std::fabs(g.wa);
    const double cw = std::fabs(g.cs2Q) + std::fabs(eb.w), ca = cw + std::fabs(g.wa * a / (3.0 * (opw + 1e-6)));
    // the features' logarithmic derivatives along a
    auto lg = [](dual x) { return x.v != 0.0 ? std::fabs(x.d / x.v) : 0.0; };
    const double la = 8.0 / a + 2.0 * lg(d.aH) + lg(d.opac) + lg(d.cs2) + lg(d.rhoQ) + 3.0 * dw / std::fabs(opw);
    for (int s = 0; s < NS; ++s) {
      const Coef<double> r0 = row_coef<double>(rd[s], eb, cx, invtau);
      const Coef<double> r1 = row_lin<NS, double>(K, s, b, g, invtau);
      const Coef<dual> d0 = row_coef<dual>(rd[s], ed, cx, invtau);
      const Coef<dual> d1 = row_lin<NS, dual>(K, s, d, gd, invtau);
      // scales: the coefficient's value, on the dark-energy rows that of its cancelling sums
      Coef<double> sc = r0;
      const uint32_t t = rd_type(rd[s]);
      if (t == R_DQ && !lambda) {
        sc.diag = 3.0 * cw * b.aH;
        sc.sup = std::fabs(opw) * (1.0 + 9.0 * ca * b.aH * b.aH / (k * k));
      }
      if (t == R_TQ && !lambda) {
        sc.diag = (1.0 + 3.0 * std::fabs(g.cs2Q)) * b.aH;
        sc.c1 = 9.0 * ca / (k * k) * std::fabs(opw) * b.aH * a * g.gde * b.rhoQ * a * a;
      }
      const double *p0 = &r0.sub, *p1 = &r1.sub, *ps = &sc.sub;
      const dual *q0 = &d0.sub, *q1 = &d1.sub;
      for (int f = 0; f < 11; ++f) {
        const double m = std::fabs(ps[f]);
        out.add(0, p1[f], p0[f], m);
        out.add(0, q1[f].v, q0[f].v, m);
        out.add(1, q1[f].d, q0[f].d, m * la);
      }
    }
  }
}

template <int NS>
int run(simt::Input &in, const char *path) {
  Params<NS> P;
  in.params<NS>(P);
  const std::vector<double> as = in.doubles(in.one<int32_t>());
  std::vector<Worst> lanes(WAVE);
  for (double k : in.k)
    for (int lam = 0; lam < 2; ++lam)
      simt::run_waves(1, [&](int) { compare<NS>(P, as, k, lam == 1, lanes[lane_id()]); });
  Worst all;
  for (const Worst &l : lanes) {
    all.n += l.n;
    for (int i = 0; i < 4; ++i) all.merge(i, l.w[i]);
  }
  FILE *out = fopen(path, "wb");
  if (!out) return 2;
  fwrite(all.w, 8, 4, out);
  fwrite(&all.n, 4, 1, out);
  fclose(out);
  return 0;
}

}  // namespace

int main(int argc, char **argv) {
  if (argc != 3) {
    fprintf(stderr, "usage: simt_rows in.bin out.bin\n");
    return 2;
  }
  simt::Input in(argv[1]);
  switch (in.layout.ns) {
    case 1: return run<1>(in, argv[2]);
    case 2: return run<2>(in, argv[2]);
    case 4: return run<4>(in, argv[2]);
    case 5: return run<5>(in, argv[2]);
    default: fprintf(stderr, "simt_rows: slot count %d not built\n", in.layout.ns); return 2;
  }
}

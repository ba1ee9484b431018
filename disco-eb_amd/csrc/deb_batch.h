// Device side of the batched solve: one workgroup per group of B consecutive k
// that share one step sequence.
#pragma once

#include "deb_forward.h"

namespace deb {

// Waves of a group's workgroup.  A group's modes are independent within a step,
// so its waves step them side by side and meet once per step for the error
// norm; one wave stepping all 16 modes of the default batch in turn left a
// launch of 8 groups on 8 of the chip's 1024 SIMDs.  Two waves per SIMD fit the
// LDS of a CU up to two slots (18 KB per wave), one wave per SIMD above
// (37 KB).  128 k in groups of 16 at lmax 11: 198 ms on one wave per group, 50.5
// ms on eight.
template <int NS>
constexpr int batch_waves() {
  return NS <= 2 ? 8 : 4;
}
// waves launched for a group of B modes: the fewest that keep the number of
// modes per wave
inline int batch_waves_of(int cap, int B) {
  const int rounds = (B + cap - 1) / cap;
  return (B + rounds - 1) / rounds;
}
// Waves of the kernel instance that runs w of them: an instance reserves the LDS
// of all its waves, so it is the smallest that holds them.  Up to four waves a
// lane has 512 registers, one wave per SIMD runs at a time, and with its waves'
// LDS a CU holds 4 / w groups.  The eight-wave instance (256 registers, spills
// at two slots) is for five waves and more, and at one slot for three and four
// too: there a wave's state is small enough that two waves per SIMD in 256
// registers beat one.  2048 groups at two slots: 2 k 5.5 ms, 4 k 11.0 ms (14.4
// and 17.9 ms on the eight-wave instance; one wave per group before the present
// step 12.2 and 24.2); at one slot 4 k 5.8 ms, on a four-wave instance 8.9.
template <int NS>
constexpr int batch_instance(int w) {
  return w <= 1 ? 1 : (w <= 2 ? 2 : (NS > 1 && w <= 4 ? 4 : 8));
}

// one wave's LDS
template <int NS>
struct BatchWave {
  double lds[fwd_lds_doubles<NS>()];
  double pcr[pcr_lds_doubles<NS>()];
  ModeU mu;
};
// what the waves of a group exchange: error sums and non-finite flags of a step
// (two sets in turn, so that one barrier per step is enough), start times
template <int NW>
struct BatchShare {
  double e2[2][NW], ts[NW];
  int bad[2][NW];
};

// orders the LDS accesses of one wave of several (they execute in order; the
// compiler must keep them so)
struct WaveSync {
  __device__ __forceinline__ void operator()() const {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
};

// evolve_modes_batched (perturbations.py:820-922) for one group of B
// consecutive k (kb .. kb + B - 1) of cosmology ci.  One step sequence serves
// the group: its start time is the minimum of the modes' start times
// (determine_start_times_per_batch :786-803) and the controller sees the RMS
// over all modes' filtered, weighted errors (rms_norm_filtered_batched
// :690-694).  Wave w of nw steps modes w, w + nw, ...; each mode's state and
// proposal live in ws (2 * NS * WAVE doubles per mode, lane-owned).  Every wave
// forms the controller's decisions from the same sums in the same order, so
// all of them take the same branches and meet at every barrier.
template <int NS, int NW>
__device__ __forceinline__ void integrate_batch(const Params<NS> &P, int ci, int kb, int B, int w, int nw,
                                                BatchWave<NS> &mine, BatchShare<NW> &sh, double *ws) {
  const int lane = lane_id();
  const BlockSync block_sync;
  const int64_t mode0 = (int64_t)ci * P.nk + kb;
  Ctx cx;
  make_ctx<NS>(cx, P, ci, P.kmodes[mode0 + w]);
  Mode<NS> m;
  m.pcr = (lds_double *)mine.pcr;
  m.u = (lds_mode_u *)&mine.mu;
#pragma unroll
  for (int s = 0; s < NS; ++s) m.rd[s] = P.rowdesc[s][lane];
  row_consts<NS>(m.rd, cx, m.rk);
  bg_init(cx, m.bg);
  m.nlev = mode_levels(P.cfg, P.nq);
  lds_double *const kl = stage_in_lds<NS>() ? (lds_double *)mine.lds : nullptr;
  auto state = [&](int b, int which) -> double * {
    return ws + ((mode0 + b) * 2 + which) * (int64_t)(NS * WAVE) + lane;
  };
  const double *tout = P.tau_out + (int64_t)ci * P.nout;
  double tmin = tout[0], tmax = tout[0];
  for (int i = 1; i < P.nout; ++i) {
    tmin = fmin(tmin, tout[i]);
    tmax = fmax(tmax, tout[i]);
  }
  double t0 = INFINITY;
  for (int b = w; b < B; b += nw) {
    cx.k = P.kmodes[mode0 + b];
    t0 = fmin(t0, start_time(cx, tmin));
  }
  if (lane == 0) sh.ts[w] = t0;
  block_sync();
  for (int i = 0; i < nw; ++i) t0 = fmin(t0, sh.ts[i]);
  const double t1 = tmax;
  for (int b = w; b < B; b += nw) {
    cx.k = P.kmodes[mode0 + b];
    double y[NS];
    initial_conditions<NS>(cx, m.rd, t0, y);
    double *dst = state(b, 0);
#pragma unroll
    for (int s = 0; s < NS; ++s) dst[s * WAVE] = y[s];
  }
  const deb_config_t &cf = P.cfg;
  const double eo = 5.0;
  const double coeff1 = (cf.icoeff + cf.pcoeff + cf.dcoeff) / eo;
  const double coeff2 = -(cf.pcoeff + 2.0 * cf.dcoeff) / eo;
  const double coeff3 = cf.dcoeff / eo;
  double tprev = t0;
  double tnext = fmin(t0 + fmin(t0 / 4.0, 0.5 * (t1 - t0)), t1);
  double prev_inv = 1.0, prev_prev_inv = 1.0;
  int iout = 0, steps = 0, set = 0, cur = 0;
  int status = DEB_STATUS_OK;
  const int width = cf.return_full ? P.n : DEB_NOUT_FIELDS;
  while (tprev < t1) {
    if (steps >= cf.max_steps) {
      status = DEB_STATUS_MAX_STEPS;
      break;
    }
    const double dt = tnext - tprev;
    double e2 = 0.0;
    bool bad = false;
    for (int b = w; b < B; b += nw) {
      const double k = P.kmodes[mode0 + b];
      cx.k = k;
      double y[NS], y1[NS], err[NS];
      const double *src = state(b, cur);
#pragma unroll
      for (int s = 0; s < NS; ++s) y[s] = src[s * WAVE];
      if (nw < B) {
        row_consts<NS>(m.rd, cx, m.rk);
        bg_set_k(m.bg, k);
      }
      rodas5_step<NS>(m, tprev, dt, y, y1, err, kl);
      // error-norm weights: indices (a, eta, delta_c, delta_b, theta_b, delta_gamma) of slot 0
      double ew = 0.0;
      if (lane == L_A || lane == L_DC || lane == L_DB || lane == L_DG) ew = 1.0;
      if (lane == L_ETA) ew = k * k;
      if (lane == L_TB) ew = 1.0 / (k * k);
      const double sc = err[0] / (cf.atol + fmax(fabs(y[0]), fabs(y1[0])) * cf.rtol);
      const double x = ew != 0.0 ? sc * ew : 0.0;
      e2 += wave_sum1(x * x);
      bad = bad || any_nonfinite<NS>(y1);
      double *dst = state(b, cur ^ 1);
#pragma unroll
      for (int s = 0; s < NS; ++s) dst[s * WAVE] = y1[s];
    }
    if (lane == 0) {
      sh.e2[set][w] = e2;
      sh.bad[set][w] = bad ? 1 : 0;
    }
    block_sync();
    double sum = 0.0;
    int any_bad = 0;
    for (int i = 0; i < nw; ++i) {
      sum += sh.e2[set][i];
      any_bad |= sh.bad[set][i];
    }
    set ^= 1;
    const double nrm = norm_or_inf(sqrt(readfirst(sum) / (6.0 * B)));
    const bool keep = nrm < 1.0;
    double inv = 1.0 / nrm;
    double fmn = keep ? 1.0 : cf.factormin;
    double factor = fmin(fmax(pid_factor(inv, prev_inv, prev_prev_inv, coeff1, coeff2, coeff3), fmn), cf.factormax);
    double dtn = dt * factor;
    if (inv == 0.0 || isinf(inv)) inv = 1.0;
    if (keep) {
      while (iout < P.nout && tout[iout] <= tnext) {
        const double th = (tout[iout] - tprev) / dt;
        for (int b = w; b < B; b += nw) {
          cx.k = P.kmodes[mode0 + b];
          const double *y0p = state(b, cur), *y1p = state(b, cur ^ 1);
          double ys[NS];
#pragma unroll
          for (int s = 0; s < NS; ++s) ys[s] = y0p[s * WAVE] + th * (y1p[s * WAVE] - y0p[s * WAVE]);
          write_outputs<NS>(P, cx, m.rd, ys, mine.lds, P.y_out + ((mode0 + b) * P.nout + iout) * (int64_t)width,
                            WaveSync());
        }
        ++iout;
      }
      prev_prev_inv = prev_inv;
      prev_inv = inv;
      cur ^= 1;  // the proposal becomes the state
      if (__builtin_amdgcn_readfirstlane(any_bad) != 0) status = DEB_STATUS_NONFINITE;
    }
    double nt0 = keep ? tnext : tprev;
    double nt1 = nt0 + dtn;
    if (nt1 > t1 - 1e-10) nt1 = keep ? t1 : nt0 + 0.5 * (t1 - nt0);
    tprev = nt0;
    tnext = nt1;
    ++steps;
    if (!keep && !(nt1 > nt0)) status = DEB_STATUS_NONFINITE;
    if (status != DEB_STATUS_OK) break;
  }
  for (int b = w; b < B; b += nw) {
    if (status != DEB_STATUS_OK)
      fill_unreached(P.y_out + (mode0 + b) * P.nout * (int64_t)width, iout, P.nout, width);
    if (lane == 0) {
      P.status[mode0 + b] = status;
      if (P.nsteps) P.nsteps[mode0 + b] = steps;
    }
  }
}

}  // namespace deb

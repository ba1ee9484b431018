"""What is timed: calls of the framework's public entry points over the range of their use.

Whole solves come in two kinds of step control, both settings of the entry points:

* adaptive at a tight tolerance (rtol 1e-9), where the returned P(k) is converged;
* a prescribed step sequence: tolerances open and the step growing by ``factormax`` from
  step to step, which makes every output a smooth function of the cosmology (what a gradient
  sampler wants) and the work of a solve a known number of steps.  Adaptive solves at loose
  tolerances take step sequences that any change of rounding alters, so that two correct
  programs agree to the tolerance only.

The rest are the single Rodas5 step, the spectra made from a solve's output fields, and the
correlation function.  Background tables are made once per process for a fixed pool of
cosmologies (a program builds them before its solves); wavenumbers, cosmologies of the pool
and cotangents come from the seed.
"""
from __future__ import annotations

import copy
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "disco-eb_amd"))

from discoeb_amd import _lib, gradient, observables, packing, tangents  # noqa: E402
from discoeb_amd.cosmology import base_theta  # noqa: E402
from discoeb_amd.perturbations import (DeviceInputs, evolve_perturbations, evolve_perturbations_batched,  # noqa: E402
                                       get_power, solve_forward)

DELTA_M = 4
POOL = 16
# hierarchies (lmaxg = lmaxgp = lmaxr, lmaxnu, nqmax) of the reference's defaults, of the
# LCDM, the massive-neutrino and the lmax-50 workloads
LAYOUTS = {11: (8, 3), 16: (8, 3), 24: (12, 4), 32: (17, 5), 50: (17, 5)}


# ---------------------------------------------------------------------------
# cases

def listed():
    return [
        # P(k) of one cosmology with the reference's default hierarchy on a few k: the smallest solve
        dict(name="pk-default-16k", kind="pk", lmax=11, nk=16, kmin=1e-4, kmax=0.1, massive=True),
        # the LCDM workload: lmax 16, no massive neutrino, 64 k
        dict(name="pk-lcdm-64k", kind="pk", lmax=16, nk=64, kmin=1e-4, kmax=0.25, massive=False),
        # one massive-neutrino cosmology, all 20 fields at 16 output times on the full k range
        dict(name="fields-mnu-256k-16out", kind="fields", lmax=32, nc=1, nk=256, kmin=1e-5, kmax=10.0, nout=16,
             growth=1.015),
        # a few cosmologies per launch: part of the chip
        dict(name="fields-5x101k-lmax24", kind="fields", lmax=24, nc=5, nk=101, kmin=1e-4, kmax=1.0, nout=1,
             growth=1.01),
        # the headline batch, P(k) arm: 64 cosmologies x 256 k in one launch
        dict(name="fields-64x256k-lmax32", kind="fields", lmax=32, nc=64, nk=256, kmin=1e-5, kmax=10.0, nout=1,
             growth=1.025),
        # groups of 16 k that share one step sequence (evolve_perturbations_batched)
        dict(name="batched-128k-by16", kind="batched", lmax=11, nk=128, batch=16, kmin=1e-4, kmax=1.0, growth=1.02),
        # P(k) and dP/dtheta: a small LCDM-sized call, the base cosmology on 256 k, many modes, lmax 50
        dict(name="grad-32k-lmax16", kind="grad", lmax=16, nc=1, nk=32, kmin=1e-4, kmax=0.5, growth=1.02),
        dict(name="grad-256k-lmax32", kind="grad", lmax=32, nc=1, nk=256, kmin=1e-5, kmax=10.0, growth=1.025),
        dict(name="grad-12x181k-lmax32", kind="grad", lmax=32, nc=12, nk=181, kmin=1e-4, kmax=1.0, growth=1.03),
        dict(name="grad-2x96k-lmax50", kind="grad", lmax=50, nc=2, nk=96, kmin=1e-4, kmax=1.0, growth=1.03),
        # one Rodas5 step of many independent states: the solver's block
        dict(name="step-1500-lmax32", kind="step", lmax=32, m=1500),
        # observables of a batch of spectra: smoothed P(k), Kaiser P(k, mu), multipoles, xi(r)
        dict(name="spectra-16x256k", kind="spectra", nc=16, nk=256, nmu=33, dlogk=0.3, ell=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pk", "fields", "batched", "grad", "grad", "step", "spectra", "spectra"])
    lmax = rng.choice([11, 16, 24, 32, 50])
    kmin = 10 ** rng.uniform(-5, -3.5)
    if kind == "pk":
        return dict(kind=kind, lmax=rng.choice([11, 16]), nk=_log_int(rng, 8, 96), kmin=kmin,
                    kmax=rng.uniform(0.03, 0.2), massive=rng.random() < 0.5)
    growth = rng.uniform(1.015, 1.04)
    if kind == "fields":
        return dict(kind=kind, lmax=lmax, nc=_log_int(rng, 1, 20), nk=_log_int(rng, 16, 256), kmin=kmin,
                    kmax=10 ** rng.uniform(-0.7, 1.0), nout=rng.choice([1, 2, 5, 16]), growth=growth)
    if kind == "batched":
        b = rng.choice([4, 7, 16])
        return dict(kind=kind, lmax=rng.choice([11, 16, 24]), nk=b * _log_int(rng, 2, 12), batch=b, kmin=kmin,
                    kmax=rng.uniform(0.1, 1.0), growth=growth)
    if kind == "grad":
        return dict(kind=kind, lmax=lmax, nc=_log_int(rng, 1, 4), nk=_log_int(rng, 16, 256), kmin=kmin,
                    kmax=10 ** rng.uniform(-0.7, 0.7), growth=max(growth, 1.025))
    if kind == "step":
        return dict(kind=kind, lmax=lmax if lmax != 50 else 32, m=_log_int(rng, 64, 2000))
    nk = 2 * _log_int(rng, 32, 512)
    # a window of at least 5 points (the smoothing polynomial is a cubic)
    return dict(kind=kind, nc=_log_int(rng, 1, 64), nk=nk, nmu=rng.choice([9, 33, 64]),
                dlogk=max(rng.uniform(0.15, 0.5), 56.0 / nk), ell=rng.choice([0, 2, 4]))


# ---------------------------------------------------------------------------
# inputs

def _pool_theta():
    """The base cosmology and its neighbours, dark energy away from the w = -1 crossing."""
    rng = np.random.default_rng(20261202)
    th = np.repeat(base_theta()[None], POOL, axis=0)
    th[1:, 0] *= rng.uniform(0.9, 1.1, POOL - 1)
    th[1:, 1] *= rng.uniform(0.95, 1.05, POOL - 1)
    th[1:, 2] += rng.uniform(-0.05, 0.05, POOL - 1)
    th[1:, 3] += rng.uniform(-0.03, 0.03, POOL - 1)
    th[1:, 5] = rng.uniform(0.04, 0.2, POOL - 1)
    th[1:, 6] = rng.uniform(-0.92, -0.85, POOL - 1)
    th[1:, 7] = rng.uniform(0.0, 0.2, POOL - 1)
    return th


@functools.lru_cache(maxsize=None)
def _pool(massive, outs):
    """(theta, param, dcosmo, dtables, dtau) of the pool's cosmologies, output times at the scale factors outs."""
    th = _pool_theta()
    if not massive:  # the LCDM workload: Lambda, no massive neutrino
        th[:, 5], th[:, 6], th[:, 7] = 0.0, -1.0, 0.0
    with np.errstate(all="ignore"):
        return (th,) + tangents.input_tangents(th, list(outs), massive_nu=massive)


def _select(param, idx):
    """The rows idx of a batched param dict."""
    out = {}
    for key, v in param.items():
        if hasattr(v, "evaluate"):
            s = copy.copy(v)
            s.x, s.y, s.S, s.I_cum, s.I_total = (a[idx] for a in (v.x, v.y, v.S, v.I_cum, v.I_total))
            out[key] = s
        elif isinstance(v, np.ndarray) and v.ndim >= 1 and v.shape[0] == POOL:
            out[key] = v[idx]
        else:
            out[key] = v
    return out


def _lm(lmax):
    lnu, nq = LAYOUTS[lmax]
    return dict(lmaxg=lmax, lmaxgp=lmax, lmaxr=lmax, lmaxnu=lnu, nqmax=nq)


def _prescribed(growth):
    return dict(rtol=1e12, atol=1e12, factormax=growth, max_steps=32768)


def _outs(case):
    n = case.get("nout", 1)
    return (1.0,) if n == 1 else tuple(float(a) for a in np.geomspace(0.01, 1.0, n))


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    dev = torch.device("cuda")
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("pk", "batched"):
        th, param = _pool(case.get("massive", True), (1.0,))[:2]
        s["param"] = _select(param, rng.integers(POOL, size=1))
        s["kmin"], s["kmax"] = case["kmin"] * rng.uniform(1.0, 1.1), case["kmax"] * rng.uniform(0.9, 1.0)
    elif kind == "fields":
        nc, nk = case["nc"], case["nk"]
        param = _pool(True, _outs(case))[1]
        p = _select(param, rng.integers(POOL, size=nc))
        cfg = packing.make_config(**_lm(case["lmax"]), **_prescribed(case["growth"]))
        k = np.geomspace(case["kmin"], case["kmax"], nk)[None, :] * rng.uniform(0.9, 1.0, size=(nc, 1))
        s.update(inp=DeviceInputs(p, cfg, dev), k=torch.from_numpy(k).to(dev),
                 tau=torch.from_numpy(packing.tau_of_aexp(p, list(_outs(case))).real.copy()).to(dev))
    elif kind == "grad":
        nc, nk = case["nc"], case["nk"]
        th, param, dcos, dtab, dtau = _pool(True, (1.0,))
        idx = rng.integers(POOL, size=nc)
        p = _select(param, idx)
        cfg = packing.make_config(**_lm(case["lmax"]), **_prescribed(case["growth"]))
        s.update(theta=th[idx], cfg=cfg, k=np.geomspace(case["kmin"], case["kmax"], nk) * rng.uniform(0.9, 1.0),
                 prepared=(DeviceInputs(p, cfg, dev), gradient.Tangents(dcos[idx], dtab[idx], dtau[idx], dev),
                           packing.tau_of_aexp(p, [1.0]).real))
    elif kind == "step":
        m = case["m"]
        param = _select(_pool(True, (1.0,))[1], rng.integers(POOL, size=1))
        lm = _lm(case["lmax"])
        n = packing.nvar(**lm)
        # states after horizon entry of modes over the k range: magnitudes of growing matter
        # perturbations, multipoles falling with l
        a = np.exp(rng.uniform(np.log(1e-4), np.log(0.9), m))
        tau = param["tau_of_a_spline"].evaluate(a[None, :])[0]
        k = np.exp(rng.uniform(np.log(1e-3), np.log(1.0), m))
        y = rng.standard_normal((m, n)) * 0.1
        y[:, 0] = a
        y[:, 3] *= 100.0
        y[:, 5] *= 100.0
        h = tau * np.exp(rng.uniform(np.log(1e-3), np.log(3e-2), m))
        T = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
        cfg = packing.make_config(**lm)
        s.update(param=param, lm=lm, inp=DeviceInputs(param, cfg, dev), cfg=cfg, kk=T(k), t0=T(tau), t1=T(tau + h),
                 y0=T(y), ci=torch.zeros(m, dtype=torch.int32, device=dev))
    else:
        nc, nk = case["nc"], case["nk"]
        k = np.geomspace(1e-4, 5.0, nk) * rng.uniform(0.9, 1.1)
        # matter transfer functions with acoustic wiggles, and the velocity field
        amp = rng.uniform(0.8, 1.2, size=(nc, 1))
        rs = rng.uniform(140.0, 155.0, size=(nc, 1))
        dm = amp * 3e5 * k**2 / (1.0 + (k / 0.015) ** 2) * np.log1p(2.0 + 30.0 * k) * (
            1.0 + 0.05 * np.sin(k * rs) * np.exp(-(k / 0.15) ** 2))
        y = rng.standard_normal((nc, nk, packing.N_OUT_FIELDS))
        y[:, :, 4] = -dm
        y[:, :, 5] = 0.5 * dm
        s.update(k=torch.from_numpy(k).to(dev), y=torch.from_numpy(y).to(dev),
                 param=dict(A_s=rng.uniform(2.0e-9, 2.2e-9, nc), n_s=rng.uniform(0.95, 0.98, nc), k_p=0.05),
                 bias=rng.uniform(1.0, 2.5, nc))
    return s


# ---------------------------------------------------------------------------
# one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "pk":
        y, k, param = evolve_perturbations(param=s["param"], aexp_out=[1.0], kmin=s["kmin"], kmax=s["kmax"],
                                           num_k=case["nk"], rtol=1e-9, atol=1e-12, max_steps=65536,
                                           **_lm(case["lmax"]))
        return get_power(k=k, y=y[:, 0], idx=DELTA_M, param=param), k
    if kind == "batched":
        y, k = evolve_perturbations_batched(param=s["param"], aexp_out=[1.0], kmin=s["kmin"], kmax=s["kmax"],
                                            num_k=case["nk"], batch_size=case["batch"], **_lm(case["lmax"]),
                                            **_prescribed(case["growth"]))
        return y, k
    if kind == "fields":
        return solve_forward(s["inp"], s["k"], s["tau"])
    if kind == "grad":
        P, G, info = gradient.power_and_gradient(s["theta"], s["k"], cfg=s["cfg"], prepared=s["prepared"])
        return P, G, info["status"], info["nsteps"]
    if kind == "step":
        inp, L = s["inp"], _lib.lib()
        y1, err = torch.empty_like(s["y0"]), torch.empty_like(s["y0"])
        p = _lib.ptr
        _lib.check(L.deb_rodas5_step(ctypes.byref(s["cfg"]), p(inp.cosmo), p(inp.tables), inp.stride, p(inp.desc),
                                     p(inp.q), p(inp.w), s["kk"].numel(), p(s["ci"]), p(s["kk"]), p(s["t0"]),
                                     p(s["t1"]), p(s["y0"]), p(y1), p(err),
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "deb_rodas5_step")
        return y1, err
    sm = observables.get_power_smoothed(k=s["k"], y=s["y"], dlogk=case["dlogk"], idx=DELTA_M, param=s["param"])
    pkmu, mu = observables.power_Kaiser(y=s["y"], kmodes=s["k"], bias=s["bias"], nmu=case["nmu"], param=s["param"],
                                        smooth_dlogk=case["dlogk"])
    p0, p2, p4 = observables.power_multipoles(y=s["y"], kmodes=s["k"], b=s["bias"], param=s["param"])
    xi, r = observables.get_xi_from_P(k=s["k"], Pk=p0, N=case["nk"], ell=case["ell"])
    return dict(smooth=sm, pkmu=pkmu, mu=mu, p0=p0, p2=p2, p4=p4, xi=xi, r=r)


# ---------------------------------------------------------------------------
# work of a pass

def _solve_steps(case):
    """Steps of a prescribed sequence (or the attempted steps an adaptive solve at rtol 1e-9 takes on average)."""
    if case["kind"] == "pk":
        return 2000.0 * (1.0 + 20.0 * case["kmax"])
    # from tau = t0 with first step t0 / 4 to 14 Gpc: t1 / t0 = 1 + (g^n - 1) / (4 (g - 1)); t0 about
    # 0.07 / k for the large k and a few Mpc for the small
    g, n = case["growth"], 0.0
    for k in np.geomspace(case["kmin"], case["kmax"], 16):
        n += math.log1p(4.0 * (g - 1.0) * 1.4e4 / min(0.07 / k, 3.0)) / math.log(g) / 16
    return n


def work(case):
    kind = case["kind"]
    if kind == "spectra":
        n = case["nc"] * case["nk"]
        w = max(4.0, case["dlogk"] * case["nk"] / 11.0)
        return dict(bytes=8.0 * n * (2 + 1 + case["nmu"] + 3 + 2) + 8.0 * case["nk"],
                    flops=n * (3 * 2 * w + 4.0 * case["nmu"] + 100 + 10.0 * math.log2(case["nk"])))
    lm = _lm(case["lmax"])
    nv = packing.nvar(**lm)
    levels = math.ceil(math.log2(case["lmax"] + 2))
    # one step: factorisation (6 values per cyclic-reduction level and row, 3 solves), 8 right-hand
    # sides of 14 and 8 solves of 5 per level + 12, 60 for the stage combinations, per state entry
    step = nv * (15.0 * levels + 11 * (5.0 * levels + 12) + 8 * 14.0 + 120)
    if kind == "step":
        return dict(bytes=8.0 * case["m"] * 3 * nv, flops=case["m"] * step)
    modes = case.get("nc", 1) * case["nk"]
    fl = modes * _solve_steps(case) * step
    by = 8.0 * modes * (1 + packing.N_OUT_FIELDS * case.get("nout", 1))
    if kind == "grad":
        fl, by = fl * 5.0, 8.0 * modes * (1 + 9 + 2 * packing.N_OUT_FIELDS)
    return dict(bytes=by, flops=fl)


# ---------------------------------------------------------------------------
# the outputs of the step and of the spectra in plain numpy / torch

def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(prepare(case, seed))
    if case["kind"] == "spectra":
        return _exact_spectra(prepare(case, seed))
    return None


class _Rows:
    """f(tau, y) = M(a, tau) y for the rows other than a (synchronous-gauge equations), the matrices of m states at
    once; complex a gives dM/da by the complex step."""

    def __init__(self, s):
        self.lm, self.k = s["lm"], s["kk"]
        p = {key: float(np.real(np.asarray(s["param"][key]).ravel()[0]))
             for key in packing.COSMO_FIELDS if key in s["param"]}
        self.p = p
        self.spl = {name: tuple(torch.from_numpy(np.ascontiguousarray(np.real(a[0]))).to(self.k.device)
                                for a in (s["param"][name].x, s["param"][name].y, s["param"][name].S))
                    for name in ("cs2a_of_loga_spline", "xe_of_loga_spline", "logrhonu_of_loga_spline")}
        self.q, self.w = packing.nu_nodes(self.lm["nqmax"])

    def spline(self, name, x):
        kx, ky, kS = self.spl[name]
        xr = x.real.contiguous()
        i = (torch.searchsorted(kx, xr) - 1).clamp(0, kx.numel() - 2)
        h = kx[i + 1] - kx[i]
        B = (x - kx[i]) / h
        A = 1.0 - B
        return A * ky[i] + B * ky[i + 1] + ((A**3 - A) * kS[i] + (B**3 - B) * kS[i + 1]) * h**2 / 6.0

    def matrix(self, a, tau):
        """(aH, M[m, n, n]) at complex scale factors a."""
        p, k, lm = self.p, self.k, self.lm
        lg, lp, lr, ln, nq = lm["lmaxg"], lm["lmaxgp"], lm["lmaxr"], lm["lmaxnu"], lm["nqmax"]
        n = packing.nvar(**lm)
        la = torch.log(a)
        rhonu = torch.exp(self.spline("logrhonu_of_loga_spline", la))
        w = p["w_DE_0"] + p["w_DE_a"] * (1.0 - a)
        rq = torch.exp(-3.0 * (1.0 + p["w_DE_0"] + p["w_DE_a"]) * la + 3.0 * (a - 1.0) * p["w_DE_a"])
        gm, gg, gr = p["grhom"], p["grhog"], p["grhor"]
        aH = torch.sqrt((gm * p["Omegam"] / a + (gg + gr * (p["Neff"] + p["Nmnu"] * rhonu)) / a**2
                         + gm * p["OmegaDE"] * rq * a**2 + gm * p["Omegak"]) / 3.0)
        cs2 = self.spline("cs2a_of_loga_spline", la) / a
        opac = self.spline("xe_of_loga_spline", la) * 2.3038921003709498e-9 * (1.0 - p["YHe"]) * p["Omegab"] * \
            p["H0"] ** 2 / a**2
        pb = 4.0 / 3.0 * gg / (gm * p["Omegab"] * a) * opac
        ca2 = w + p["w_DE_a"] * a / 3.0 / (1.0 + w + 1e-6)
        cq = p["cs2_DE"]
        dens = gm * p["OmegaDE"] * rq * a**2
        M = torch.zeros((a.numel(), n, n), dtype=a.dtype, device=a.device)
        fh, fe, fp = (torch.zeros((a.numel(), n), dtype=a.dtype, device=a.device) for _ in range(3))
        f1 = torch.zeros_like(fh)
        ig, ip, ir, iq = 7, 8 + lg, 9 + lg + lp, 10 + lg + lp + lr
        k2 = k * k
        oc, ob = p["Omegam"] - p["Omegab"], p["Omegab"]
        # h', eta', Pi and the source of (a h')' as linear functionals of the state
        fh[:, 2] = 2 * k2 / aH
        for i, rho in ((3, gm * oc / a), (5, gm * ob / a), (ig, gg / a**2), (ir, gr * p["Neff"] / a**2), (n - 2, dens)):
            fh[:, i] = rho / aH
        f1[:, 3], f1[:, 5] = -gm * oc, -gm * ob
        f1[:, ig], f1[:, ir] = -2.0 * gg / a, -2.0 * gr * p["Neff"] / a
        f1[:, n - 2] = -a * dens * (1.0 + 3.0 * cq)
        f1[:, n - 1] = -a * 9.0 * (cq - ca2) * aH / k2 * (1.0 + w) * dens
        for i, rho in ((4, gm * oc / a), (6, gm * ob / a), (ig + 1, 4.0 / 3.0 * gg / a**2),
                       (ir + 1, 4.0 / 3.0 * gr * p["Neff"] / a**2), (n - 1, (1.0 + w) * dens)):
            fe[:, i] = rho / (2 * k2)
        v = [1.0 / torch.sqrt(1.0 + (a * p["amnu"] / q) ** 2) for q in self.q]
        rn = gr * p["Nmnu"] / a**2
        for j in range(nq):
            fh[:, iq + j] = rn * self.w[j] / v[j] / aH
            f1[:, iq + j] = -rn * a * self.w[j] * (1.0 / v[j] + v[j])
            fe[:, iq + nq + j] = rn * k * self.w[j] / (2 * k2)
        fp[:, ig + 2] = fp[:, ip] = fp[:, ip + 2] = 1.0

        def add(i, j, c):
            M[:, i, j] += c

        def enter(i, h=0.0, e=0.0, pi=None):
            M[:, i] += h * fh + e * fe
            if pi is not None:
                M[:, i] += pi[:, None] * fp
        M[:, 1] = f1
        enter(2, e=1.0)
        add(3, 4, -1.0), enter(3, h=-0.5), add(4, 4, -aH)
        add(5, 6, -1.0), enter(5, h=-0.5)
        add(6, 5, k2 * cs2), add(6, 6, -aH - pb), add(6, ig + 1, pb)
        add(ig, ig + 1, -4.0 / 3.0), enter(ig, h=-2.0 / 3.0)
        add(ig + 1, ig, k2 / 4.0), add(ig + 1, ig + 2, -k2 / 2.0), add(ig + 1, ig + 1, -opac), add(ig + 1, 6, opac)
        add(ig + 2, ig + 1, 8.0 / 15.0), add(ig + 2, ig + 3, -0.6 * k), add(ig + 2, ig + 2, -opac)
        enter(ig + 2, h=4.0 / 15.0, e=8.0 / 5.0, pi=0.1 * opac)
        for lx, i0, first in ((lg, ig, 3), (lp, ip, 1)):
            for l in range(first, lx):  # noqa: E741
                add(i0 + l, i0 + l - 1, k * l / (2 * l + 1)), add(i0 + l, i0 + l + 1, -k * (l + 1) / (2 * l + 1))
                add(i0 + l, i0 + l, -opac)
            add(i0 + lx, i0 + lx - 1, k), add(i0 + lx, i0 + lx, -(lx + 1) / tau - opac)
        add(ip, ip + 1, -k), add(ip, ip, -opac), enter(ip, pi=0.5 * opac), enter(ip + 2, pi=0.1 * opac)
        add(ir, ir + 1, -4.0 / 3.0), enter(ir, h=-2.0 / 3.0)
        add(ir + 1, ir, k2 / 4.0), add(ir + 1, ir + 2, -k2 / 2.0)
        add(ir + 2, ir + 1, 8.0 / 15.0), add(ir + 2, ir + 3, -0.6 * k), enter(ir + 2, h=4.0 / 15.0, e=8.0 / 5.0)
        for l in range(3, lr):  # noqa: E741
            add(ir + l, ir + l - 1, k * l / (2 * l + 1)), add(ir + l, ir + l + 1, -k * (l + 1) / (2 * l + 1))
        add(ir + lr, ir + lr - 1, k), add(ir + lr, ir + lr, -(lr + 1) / tau)
        for j in range(nq):
            dl = -self.q[j] / (1.0 + math.exp(-self.q[j]))
            kv, at = k * v[j], lambda l: iq + l * nq + j  # noqa: E731
            add(at(0), at(1), -kv), enter(at(0), h=dl / 6.0)
            for l in range(1, ln):  # noqa: E741
                add(at(l), at(l - 1), kv * l / (2 * l + 1)), add(at(l), at(l + 1), -kv * (l + 1) / (2 * l + 1))
            enter(at(2), h=-dl / 15.0, e=-0.4 * dl)
            add(at(ln), at(ln - 1), kv), add(at(ln), at(ln), -(ln + 1) / tau)
        add(n - 2, n - 2, -3.0 * (cq - w) * aH)
        add(n - 2, n - 1, -(1.0 + w) - 9.0 * (1.0 + w) * (cq - ca2) * aH**2 / k2)
        M[:, n - 2] += (-0.5 * (1.0 + w))[:, None] * fh
        add(n - 1, n - 2, cq / (1.0 + w) * k2), add(n - 1, n - 1, -(1.0 - 3.0 * cq) * aH)
        return aH, M

    def rhs(self, tau, y):
        aH, M = self.matrix(y[:, 0].to(torch.complex128), tau)
        f = (M.real @ y[:, :, None])[:, :, 0]
        f[:, 0] = aH.real * y[:, 0]
        return f


def _exact_step(s):
    """Rodas5 in its transformed form: dense Jacobian, dense solves."""
    m = s["kk"].numel()
    out = []
    for lo in range(0, m, 256):
        part = dict(s, kk=s["kk"][lo:lo + 256])
        out.append(_exact_steps(_Rows(part), *(s[x][lo:lo + 256] for x in ("t0", "t1", "y0"))))
    return tuple(torch.cat(x) for x in zip(*out))


def _exact_steps(rows, t0, t1, y0):
    A = ((), (2.0,), (3.040894194418781, 1.041747909077569),
         (2.576417536461461, 1.622083060776640, -0.9089668560264532),
         (2.760842080225597, 1.446624659844071, -0.3036980084553738, 0.2877498600325443),
         (-14.09640773051259, 6.925207756232704, -41.47510893210728, 2.343771018586405, 24.13215229196062))
    A = A + (A[5] + (1.0,), A[5] + (1.0, 1.0))
    C = ((), (-10.31323885133993,), (-21.04823117650003, -7.234992135176716),
         (32.22751541853323, -4.943732386540191, 19.44922031041879),
         (-20.69865579590063, -8.816374604402768, 1.260436877740897, -0.7495647613787146),
         (-46.22004352711257, -17.49534862857472, -289.6389582892057, 93.60855400400906, 318.3822534212147),
         (34.20013733472935, -14.15535402717690, 57.82335640988400, 25.83362985412365, 1.408950972071624,
          -6.551835421242162),
         (42.57076742291101, -13.80770672017997, 93.98938432427124, 18.77919633714503, -31.58359187223370,
          -6.685968952921985, -5.810979938412932))
    c = (0.0, 0.38, 0.3878509998321533, 0.4839718937873840, 0.4570477008819580, 1.0, 1.0, 1.0)
    d = (0.19, -0.1823079225333714636, -0.319231832186874912, 0.3449828624725343, -0.377417564392089818, 0.0, 0.0, 0.0)
    eps = 1e-30
    h = t1 - t0
    a = torch.complex(y0[:, 0], torch.full_like(t0, eps))
    aH, M = rows.matrix(a, t0)
    J = M.real.clone()
    J[:, :, 0] += (M.imag @ y0[:, :, None])[:, :, 0] / eps
    J[:, 0, 0] = (aH * a).imag / eps
    # only the truncation rows depend on tau: -(l + 1) / tau on their diagonals
    lm = rows.lm
    lg, lp, lr, ln, nq = lm["lmaxg"], lm["lmaxgp"], lm["lmaxr"], lm["lmaxnu"], lm["nqmax"]
    dT = torch.zeros_like(y0)
    last = [(7 + lg, lg), (8 + lg + lp, lp), (9 + lg + lp + lr, lr)]
    last += [(10 + lg + lp + lr + ln * nq + j, ln) for j in range(nq)]
    for i, l in last:  # noqa: E741
        dT[:, i] = (l + 1) / t0**2 * y0[:, i]
    W = -J
    W.diagonal(dim1=1, dim2=2).add_((1.0 / (0.19 * h))[:, None])
    LU, piv = torch.linalg.lu_factor(W)
    ks = []
    for i in range(8):
        u = y0 + sum((x * kj for x, kj in zip(A[i], ks)), torch.zeros_like(y0))
        r = rows.rhs(t0 + c[i] * h, u) + d[i] * h[:, None] * dT
        r = r + sum((x / h[:, None] * kj for x, kj in zip(C[i], ks)), torch.zeros_like(y0))
        ks.append(torch.linalg.lu_solve(LU, piv, r[:, :, None])[:, :, 0])
    return u + ks[7], ks[7]


def _exact_spectra(s):
    from scipy.special import loggamma
    case = s["case"]
    k, y = s["k"].cpu().numpy(), s["y"].cpu().numpy()
    A_s, n_s = (s["param"][x][:, None] for x in ("A_s", "n_s"))
    prim = 2 * np.pi**2 * A_s * (k / 0.05) ** (n_s - 1.0) * k**-3
    W = int(np.round(case["dlogk"] / (np.log(k[1]) - np.log(k[0]))))
    W += (W + 1) % 2
    # least-squares cubic through W points, value at the centre
    x = (np.arange(W) - W // 2) / max(W // 2, 1)
    q, r = np.linalg.qr(np.vander(x, 4, increasing=True))
    c = q @ np.linalg.solve(r.T, np.eye(4)[0])

    def smooth(P):
        out = np.exp(np.array([np.convolve(v, c, mode="same") for v in np.log(P)]))
        out[:, :W // 2], out[:, -((W + 1) // 2):] = P[:, :W // 2], P[:, -((W + 1) // 2):]
        return out
    pd, pt = prim * y[:, :, 4] ** 2, prim * y[:, :, 5] ** 2
    sd, st = smooth(pd), smooth(pt)
    mu = np.linspace(-1, 1, case["nmu"])
    b = s["bias"][:, None]
    pkmu = (b[:, :, None] * np.sqrt(sd)[:, :, None] + mu**2 * np.sqrt(st)[:, :, None]) ** 2
    f = np.sqrt(prim)
    dl, th = f * y[:, :, 4], f * y[:, :, 5]
    p0 = b**2 * dl**2 - 2 * b / 3 * dl * th + th**2 / 5
    p2 = -4 * b / 3 * dl * th + 4.0 / 7.0 * th**2
    p4 = 8.0 / 35.0 * th**2
    n, ell = case["nk"], case["ell"]
    kap = np.pi * np.arange(n // 2 + 1) / np.log(k[-1] / k[0])
    ph = loggamma((1.5 + ell) / 2 + 1j * kap).imag - np.log(np.pi) * kap
    g = np.fft.irfft(np.fft.rfft(p0 * k**1.5, axis=1) * np.exp(2j * ph), n, axis=1)
    rr = 2 * np.pi / k
    xi = ((1j**ell).real * g / (2 * np.pi * rr) ** 1.5)[:, ::-1]
    T = lambda v: torch.from_numpy(np.ascontiguousarray(v))  # noqa: E731
    return dict(smooth=T(sd), pkmu=T(pkmu), mu=T(mu), p0=T(p0), p2=T(p2), p4=T(p4), xi=T(xi),
                r=T(np.broadcast_to(rr[::-1], (case["nc"], n))))

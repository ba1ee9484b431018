"""The right-hand side and the Rodas5 step against the oracle where their lane
layouts and tables have edges: every slot count, chains of 32 and 33 rows (the
last cyclic-reduction level starts at 33), massive-neutrino chains in slot 0,
and log a on, between and outside the splines' knots."""
import numpy as np
import pytest

import oracle
from discoeb_amd import packing
from discoeb_amd.perturbations import DeviceInputs
from test_gpu_parity import _hook, _states

pytestmark = pytest.mark.gpu

# (lmaxg, lmaxgp, lmaxr, lmaxnu, nqmax): slots
LAYOUTS = [(3, 3, 3, 3, 0), (4, 3, 5, 3, 2), (30, 31, 31, 3, 1), (31, 32, 32, 31, 2), (15, 17, 62, 32, 1),
           (54, 63, 63, 5, 3), (20, 40, 33, 34, 3), (50, 50, 50, 33, 3)]


def _prob(param, lay):
    cfg = packing.make_config(lmaxg=lay[0], lmaxgp=lay[1], lmaxr=lay[2], lmaxnu=lay[3], nqmax=lay[4])
    return cfg, oracle.Problem(param, cfg), DeviceInputs(param, cfg)


def _check_rhs(prob, k, tau, y, f):
    ref = prob.rhs(k, tau, y)
    J, _ = prob.jacobian(k, tau, y)
    scale = np.abs(J) @ np.abs(y) + np.abs(ref)
    assert np.all(np.abs(f - ref) <= 1e-13 * scale + 1e-300), (k, tau)


@pytest.mark.parametrize("lay", LAYOUTS)
def test_layout_edges(gpu, test_param, lay):
    cfg, prob, inp = _prob(test_param, lay)
    kk = np.array([3e-4, 0.2, 5.0])
    taus, ys = _states(prob, test_param, kk, seed=5)
    f = _hook("rhs", cfg, inp, kk, taus, ys)
    hs = taus * np.array([0.1, 0.05, 0.01])
    y1, err = _hook("step", cfg, inp, kk, taus, ys, taus + hs)
    for i, k in enumerate(kk):
        _check_rhs(prob, k, taus[i], ys[i], f[i])
        r1, re = prob.rodas5_step(k, taus[i], taus[i] + hs[i], ys[i])
        sc = np.abs(r1) + np.abs(ys[i]) + np.abs(re) + 1e-300
        assert (np.abs(y1[i] - r1) / sc).max() < 1e-9, k


def test_background_table_edges(gpu, test_param):
    cfg, prob, inp = _prob(test_param, (11, 11, 11, 8, 3))
    x = test_param["xe_of_loga_spline"].x
    x = np.real(np.asarray(x)).reshape(-1, x.shape[-1])[0]
    n = x.size
    la = np.concatenate([x[[0, 1, 15, 16, 17, n // 2, n - 17, n - 2]], 0.5 * (x[[0, 16, n - 3, n - 2]] + x[[1, 17, n - 2, n - 1]]),
                         [x[0] - 1e-3, x[-1] - 1e-12]])
    kk = np.full(la.size, 0.05)
    taus, ys = _states(prob, test_param, kk, seed=6)
    ys[:, 0] = np.exp(la)
    f = _hook("rhs", cfg, inp, kk, taus, ys)
    for i in range(la.size):
        _check_rhs(prob, kk[i], taus[i], ys[i], f[i])

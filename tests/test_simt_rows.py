"""The coefficients that the kernels' right-hand sides run (rows as per-mode
constants times background features, the background from register-held spline
windows), on the CPU under the sanitizers, row by row against the equations
(row_coef) and against the plain background, in doubles and along a, with and
without the dark-energy fluid.

Bounds in units of 2^-52: a row is a product or sum of at most 14 roundings on
either side, 16 of its value (on the dark-energy rows of its cancelling terms);
a derivative sums such products over its features' derivatives, 64.  The
background's scales hold its rounding already: 1."""
import subprocess

import numpy as np
import pytest

import oracle
from discoeb_amd import packing
from test_simt_host import AOUT, SIMT, _finish, _start, _write

LAYOUTS = {"ns1-nu": dict(lmaxg=4, lmaxgp=3, lmaxr=5, lmaxnu=3, nqmax=2),
           "ns1-massless": dict(lmaxg=16, lmaxgp=16, lmaxr=16, lmaxnu=8, nqmax=0),
           "ns2": dict(lmaxg=11, lmaxgp=11, lmaxr=11, lmaxnu=8, nqmax=3),
           "ns4": dict(lmaxg=32, lmaxgp=32, lmaxr=32, lmaxnu=17, nqmax=5),
           "ns5": dict(lmaxg=50, lmaxgp=50, lmaxr=50, lmaxnu=17, nqmax=5)}
BOUNDS = (16.0, 64.0, 1.0, 1.0)


@pytest.fixture(scope="module")
def rows():
    r = subprocess.run(["make", "-C", SIMT, "simt_rows"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    return SIMT + "/simt_rows"


def _scale_factors(param):
    """Forwards over the splines' range, backwards over it, and back and forth between neighbouring windows; on a
    knot, outside the knots on both sides, at a = 1."""
    x = np.real(np.asarray(param["xe_of_loga_spline"].x)).reshape(-1, param["xe_of_loga_spline"].x.shape[-1])[0]
    up = np.geomspace(np.exp(x[0]) * 0.9, 1.0, 14)
    i = x.size // 2
    near = np.exp([x[i], x[i + 12], x[i + 13] + 1e-9, x[i - 3] - 1e-9, x[i - 4], x[-2], x[-1] + 1e-3])
    return np.concatenate([up, up[::-3], near])


def test_rows_and_background(rows, test_param, grad_inputs, tmp_path):
    procs = {}
    for name, lay in LAYOUTS.items():
        # the gradient inputs: w0 and wa of a fluid, massive neutrinos; two layouts on the test cosmology
        param = test_param if name in ("ns2", "ns1-massless") else grad_inputs["param"]
        cfg = packing.make_config(**lay)
        a = _scale_factors(param)
        extra = np.int32(a.size).tobytes() + a.tobytes()
        _write(tmp_path / f"{name}.in", 0, cfg, oracle.Problem(param, cfg), np.array([1e-4, 2.0]),
               packing.tau_of_aexp(param, AOUT)[0], extra)
        procs[name] = _start(rows, tmp_path, name)
    for name, p in procs.items():
        _finish(p, 900)
        raw = (tmp_path / f"{name}.out").read_bytes()
        worst, n = np.frombuffer(raw[:32]), np.frombuffer(raw[32:], np.int32)[0]
        assert n > 0 and np.all(worst <= BOUNDS), (name, worst)

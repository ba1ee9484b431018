"""The batched solve's device code (integrate_batch) on the CPU under the
sanitizers, several waves per group: 64 host threads per wave, the workgroup
barrier over all of them (a wave that left the step loop alone would never
complete it; the run's time limit catches that).  Prescribed large steps, so
that a group ends within a few of them; the oracle takes the same steps."""
import subprocess

import numpy as np
import pytest

import oracle
from discoeb_amd import packing
from test_simt_host import SIMT, _finish, _start, _write

NS1 = dict(lmaxg=4, lmaxgp=3, lmaxr=5, lmaxnu=3, nqmax=2)
NS5 = dict(lmaxg=50, lmaxgp=50, lmaxr=50, lmaxnu=17, nqmax=5)  # stage vectors in registers
AOUT = [2e-5, 1e-4]
K3 = np.geomspace(2e-3, 2e-2, 3)


@pytest.fixture(scope="module")
def batch():
    r = subprocess.run(["make", "-C", SIMT, "simt_batch"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    return SIMT + "/simt_batch"


def _prescribed(**kw):
    return dict(dict(rtol=1e12, atol=1e12, factormax=3.0, factormin=1e-6, max_steps=64), **kw)


# name: (layout, k, batch, waves, configuration)
RUNS = {
    # uneven last round, one mode per wave, two groups
    "uneven": (NS1, K3, 3, 2, _prescribed()),
    "full": (NS1, K3, 3, 3, _prescribed()),
    "pairs": (NS1, np.geomspace(2e-3, 2e-2, 4), 2, 2, _prescribed()),
    "registers": (NS5, K3[:2], 2, 2, _prescribed()),
    # the step limit between the two output times
    "limit": (NS1, K3, 3, 2, _prescribed(max_steps=4)),
    # a mode of the second wave without finite values: every step is rejected
    "nonfinite": (NS1, np.array([2e-3, np.nan, 2e-2]), 3, 2, _prescribed()),
}


def test_groups_of_several_waves(batch, test_param, tmp_path):
    tau = packing.tau_of_aexp(test_param, AOUT)[0]
    runs = {}
    for name, (lay, k, B, nw, conf) in RUNS.items():
        cfg = packing.make_config(**lay, **conf)
        prob = oracle.Problem(test_param, cfg)
        _write(tmp_path / f"{name}.in", 0, cfg, prob, k, tau, np.int32(B).tobytes() + np.int32(nw).tobytes())
        runs[name] = (prob, k, B, cfg.max_steps, _start(batch, tmp_path, name))
    for name, (prob, k, B, max_steps, p) in runs.items():
        _finish(p, 900)
        raw = (tmp_path / f"{name}.out").read_bytes()
        st, ns = np.frombuffer(raw[:8 * k.size], np.int32).reshape(2, k.size)
        y = np.frombuffer(raw[8 * k.size:]).reshape(k.size, len(AOUT), 20)
        ref = prob.evolve_batched(k, tau, B, nthreads=2)
        assert np.array_equal(st, ref["status"]) and np.array_equal(ns, ref["nsteps"]), (name, st, ns, ref)
        if name == "limit":
            assert np.all(st == packing.STATUS_MAX_STEPS) and np.all(ns == max_steps)
        elif name == "nonfinite":
            assert np.all(st == packing.STATUS_NONFINITE)
        else:
            assert np.all(st == packing.STATUS_OK)
        reached = np.isfinite(ref["y"]).all(axis=2)
        assert np.array_equal(np.isfinite(y).all(axis=2), reached) and np.all(np.isposinf(y[~reached])), name
        if name == "limit":
            assert np.all(reached == [True, False])
        for f in (4, 6, 8, 10, 12):
            assert np.all(np.abs(y[reached][:, f] / ref["y"][reached][:, f] - 1) < 1e-8), (name, f)

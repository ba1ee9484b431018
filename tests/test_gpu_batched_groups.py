"""Groups of the batched solve on the instances of one, two, four and eight
waves, several cosmologies in one launch, against the oracle's restatement on
prescribed steps (open tolerances, the step growing by factormax)."""
import numpy as np
import pytest

import oracle
from discoeb_amd import packing
from discoeb_amd.background import evolve_background
from discoeb_amd.cosmology import base_theta, param_from_theta
from discoeb_amd.perturbations import DeviceInputs, solve_forward
from test_gpu_batched import SMALL
from test_gpu_batched_waves import LARGE

pytestmark = pytest.mark.gpu


def _theta(i):
    th = base_theta()[None].copy()
    th[0, 0] *= 1.0 + 0.03 * i
    return th


def _param(th):
    with np.errstate(all="ignore"):
        return evolve_background(param=param_from_theta(th))


@pytest.fixture(scope="module")
def two():
    """Two cosmologies: the batched tables and each one's own."""
    th = np.concatenate([_theta(0), _theta(1)])
    return _param(th), [_param(th[i:i + 1]) for i in range(2)]


def _solve(param, cfg, k, tau, batch):
    import torch
    y, st, ns = solve_forward(DeviceInputs(param, cfg), torch.from_numpy(k), torch.from_numpy(tau), throw=False,
                              batch_size=batch)
    return y.cpu().numpy(), st.cpu().numpy(), ns.cpu().numpy()


def _inputs(two, cfg, nk, aout):
    tau = np.stack([packing.tau_of_aexp(p, aout)[0].real for p in two[1]])
    k = np.geomspace(1e-3, 0.1, nk)[None] * np.array([[1.0], [1.07]])
    return np.ascontiguousarray(k), np.ascontiguousarray(tau)


@pytest.mark.parametrize("lay,batch", [(SMALL, 1), (SMALL, 2), (SMALL, 4), (SMALL, 6), (LARGE, 1), (LARGE, 3)])
def test_cosmologies_and_instances(gpu, two, lay, batch):
    cfg = packing.make_config(rtol=1e12, atol=1e12, factormax=1.15, max_steps=4096, **lay)
    k, tau = _inputs(two, cfg, 3 * batch, [0.02, 0.1])
    y, st, ns = _solve(two[0], cfg, k, tau, batch)
    assert np.all(st == 0)
    for c, p in enumerate(two[1]):
        ref = oracle.Problem(p, cfg).evolve_batched(k[c], tau[c], batch, nthreads=8)
        assert np.all(ref["status"] == 0) and np.array_equal(ns[c], ref["nsteps"])
        for f in (4, 6, 8, 10, 12):
            assert np.abs(y[c, :, :, f] / ref["y"][:, :, f] - 1).max() < 1e-8, (c, f)


@pytest.mark.parametrize("lay,batch", [(SMALL, 2), (SMALL, 9), (SMALL, 16), (LARGE, 5)])
def test_groups_that_reach_the_step_limit(gpu, two, lay, batch):
    """A limit that some groups end below and others reach between two outputs: every mode of a group has the group's
    status and step count, unreached outputs hold inf, what was reached is the unlimited run's to the bit."""
    conf = dict(rtol=1e12, atol=1e12, factormax=1.15)
    cfg = packing.make_config(max_steps=4096, **conf, **lay)
    k, tau = _inputs(two, cfg, 3 * batch, [0.02, 0.1])
    y, st, ns = _solve(two[0], cfg, k, tau, batch)
    assert np.all(st == 0)
    limit = int(ns.max()) - 1
    assert limit > ns.min()
    cfg = packing.make_config(max_steps=limit, **conf, **lay)
    yl, sl, nl = _solve(two[0], cfg, k, tau, batch)
    over = ns > limit
    assert np.array_equal(sl, np.where(over, packing.STATUS_MAX_STEPS, packing.STATUS_OK))
    assert np.array_equal(nl, np.minimum(ns, limit))
    assert np.array_equal(yl[~over], y[~over])
    assert np.array_equal(yl[over][:, 0], y[over][:, 0]) and np.all(np.isposinf(yl[over][:, 1]))


@pytest.mark.parametrize("lay,batch,bad", [(SMALL, 2, 1), (SMALL, 4, 2), (SMALL, 9, 3), (SMALL, 16, 15), (LARGE, 5, 4)])
def test_group_with_a_nonfinite_mode(gpu, two, lay, batch, bad):
    """A mode of a wave other than the first without finite values rejects every step of its group until the step no
    longer advances; the other groups are unchanged to the bit."""
    cfg = packing.make_config(rtol=1e12, atol=1e12, factormax=1.15, factormin=1e-6, max_steps=4096, **lay)
    k, tau = _inputs(two, cfg, 3 * batch, [0.02, 0.1])
    y, st, _ = _solve(two[0], cfg, k, tau, batch)
    assert np.all(st == 0)
    kb = k.copy()
    kb[1, batch + bad] = np.nan
    yb, sb, nb = _solve(two[0], cfg, kb, tau, batch)
    hit = np.zeros(k.shape, bool)
    hit[1, batch:2 * batch] = True
    ref = oracle.Problem(two[1][1], cfg).evolve_batched(kb[1, batch:2 * batch], tau[1], batch, nthreads=2)
    assert np.array_equal(sb[hit], ref["status"]) and np.array_equal(nb[hit], ref["nsteps"])
    assert np.all(sb[hit] == packing.STATUS_NONFINITE) and np.all(np.isposinf(yb[hit]))
    assert np.all(sb[~hit] == 0) and np.array_equal(yb[~hit], y[~hit])

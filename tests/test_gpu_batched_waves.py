"""Groups of the batched solve over the sizes where their split over a
workgroup's waves changes: fewer modes than waves, an uneven last round, more
than two rounds, and both wave counts (two and four slots).  Each against the
oracle's restatement on prescribed steps (open tolerances, the step growing by
factormax), where every output is a smooth function of the rounding."""
import numpy as np
import pytest

import oracle
from discoeb_amd import packing
from test_gpu_batched import SMALL, _gpu

pytestmark = pytest.mark.gpu

LARGE = dict(lmaxg=32, lmaxgp=32, lmaxr=32, lmaxnu=17, nqmax=5)


@pytest.mark.parametrize("lay,batch,groups", [(SMALL, 1, 3), (SMALL, 3, 2), (SMALL, 8, 1), (SMALL, 9, 2),
                                              (SMALL, 17, 1), (LARGE, 2, 1), (LARGE, 5, 1)])
def test_group_sizes(gpu, test_param, lay, batch, groups):
    cfg = packing.make_config(rtol=1e12, atol=1e12, factormax=1.15, max_steps=4096, **lay)
    k = np.geomspace(1e-3, 0.1, batch * groups)
    tau = packing.tau_of_aexp(test_param, [0.02, 0.1])[0]
    y, st, ns = _gpu(test_param, cfg, k, tau, batch)
    ref = oracle.Problem(test_param, cfg).evolve_batched(k, tau, batch, nthreads=8)
    assert np.all(st == 0) and np.all(ref["status"] == 0)
    assert np.array_equal(ns, ref["nsteps"])
    for f in (4, 6, 8, 10, 12):
        scale = np.abs(ref["y"][:, :, f])
        assert (np.abs(y[:, :, f] - ref["y"][:, :, f]) / scale).max() < 1e-8, f

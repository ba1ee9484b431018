"""Smoothing windows and transform lengths at the edges of the observables'
kernels: windows of fewer and of more points than a wavefront's lanes, the
shortest and the longest transform.  The smoothing coefficients are formed
here in exact fractions: the oracle's least-squares solve of the unscaled
Vandermonde system is off by 1.5e-13 at 65 points and 2.4e-11 at 1001 (sum of
the coefficients' errors), which log P multiplies by about ten."""
from fractions import Fraction

import numpy as np
import pytest

import observables as ob
from test_gpu_observables import _inputs, _p

pytestmark = pytest.mark.gpu


def _cubic_coeffs(W):
    """The symmetric cubic filter's closed form: c_j = (a - b x_j^2) with the moments of x = -h..h."""
    h = W // 2
    x2 = [Fraction((h - j) ** 2) for j in range(W)]
    s0, s2, s4 = Fraction(W), sum(x2), sum(v * v for v in x2)
    det = s0 * s4 - s2 * s2
    return np.array([float((s4 - s2 * v) / det) for v in x2])


@pytest.mark.parametrize("nk,W", [(64, 5), (256, 63), (256, 65), (512, 131), (2048, 1001)])
def test_window_lengths(gpu, nk, W):
    from discoeb_amd import observables as gob
    k, y, param = _inputs(B=2, nk=nk)
    dlogk = W * (np.log(k[1]) - np.log(k[0]))
    assert gob._window_length(k, dlogk) == W
    got = gob.get_power_smoothed(k=k, y=y, dlogk=dlogk, idx=4, param=param).cpu().numpy()
    for b in range(2):
        P = ob.power(k, y[b], 4, *_p(param, b))
        want = np.exp(np.convolve(np.log(P), _cubic_coeffs(W), mode="same"))
        want[:W // 2], want[-((W + 1) // 2):] = P[:W // 2], P[-((W + 1) // 2):]
        np.testing.assert_allclose(got[b], want, rtol=1e-12)


@pytest.mark.parametrize("N", [2, 4, 254, 258, 2048])
def test_transform_lengths(gpu, N):
    from discoeb_amd import observables as gob
    k = np.geomspace(1e-4, 10.0, N)
    Pk = (k * np.exp(-(k * 5) ** 2))[None] * np.array([[1.0], [2.0]])
    xi, r = (t.cpu().numpy() for t in gob.get_xi_from_P(k=k, Pk=Pk, N=N, ell=0))
    for b in range(2):
        want, r_ref = ob.xi_from_P(k, Pk[b], 0)
        np.testing.assert_allclose(r[b], r_ref, rtol=1e-15)
        np.testing.assert_allclose(xi[b], want, rtol=0, atol=1e-11 * np.abs(want).max() + 1e-300)

"""The FP64 flux by two lanes per face (csrc/gkm_pair.hpp) where its exchange and
its own exp and square root can go wrong: face counts around the 32 faces of a
wave, and collision times far below and above dt (exp(-dt/tau) from 0 to 1).

Tolerance against the oracle: 1e-12 of each component's largest magnitude, the
bound of the flux batch everywhere in this suite (about 5000 FP64 roundings of
terms that do not exceed the result by more than 1e1).  For dt << tau the time
coefficients dt - tau (1 - e^(-dt/tau)) and dt e - tau (1 - e) cancel to
(dt/tau)/2 of their terms, which is then divided out (GKMflux.cpp:162-167): an
error of one ulp there reads 2 tau/dt times as large, so the bound is
max(1e-12, 40 eps tau/dt); the flux depends on them through the slope terms
alone, which are below its Euler part."""
import numpy as np
import pytest

import pyoracle as po
from cases import make_case, random_faces
from dns_gkm_lpt_amd import _lib as gl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 65])
@pytest.mark.parametrize("ratio", [1e-3, 1.0, 50.0, 1e4])  # dt/tau of the smooth part
def test_pair_flux_matches_oracle(n, ratio):
    W, P, gas = make_case(32)
    X = random_faces(n, seed=11 + n)
    tau = np.array([po.tau_of(X[i, :5], gas) for i in range(n)])
    dt = float(ratio * tau[0])
    ref = po.flux(X, tau, dt, gas)
    with gl.Context(32, P) as c:
        F = c.flux_batch(X, tau, dt)
    scale = np.max(np.abs(ref), axis=0)
    tol = max(1e-12, 40 * np.finfo(float).eps / ratio)
    assert np.all(np.max(np.abs(F - ref), axis=0) <= tol * scale), (F - ref) / scale


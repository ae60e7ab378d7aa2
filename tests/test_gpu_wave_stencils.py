"""Stencils of the 5..32-band kernels around their load batches (12, 6 and 4 rows) and
band counts whose packed elements end inside a wave or between two: random tables
against the oracle, one right-hand side and two RK4 steps."""
import numpy as np
import pytest

from helpers import N
from test_gpu_small_terms import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nn,nk", [(5, 13, 17), (6, 0, 9), (6, 12, 40), (7, 1, 8), (8, 11, 33), (8, 25, 20), (8, 64, 15), (13, 7, 11), (14, 6, 12),
                                      (17, 5, 6), (18, 4, 7), (24, 9, 6), (31, 3, 5)])
def test_stencil_batches_match_oracle(nb, nn, nk):
    p, t, osys = _problem(nb, nk, nn, nb % 2 == 0, 2, N.STEPPER_RK4, 4, 100 * nb + nn)
    eng = N.Engine(p)
    f = 0.3 * np.random.default_rng(nn).normal(size=(2, 3, 6))
    got, ref = eng.rhs(f[0, 0]), osys.rhs(t["P"], f[0, 0], True)
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))  # the suite's bar for right-hand sides
    P, dt = t["P"], 0.01
    for E in f:
        k1 = osys.rhs(P, E[0], True)
        k2 = osys.rhs(P + dt / 2 * k1, E[1], True)
        k3 = osys.rhs(P + dt / 2 * k2, E[1], True)
        P = P + dt / 6 * (k1 + 2 * k2 + 2 * k3 + osys.rhs(P + dt * k3, E[2], True))
    eng.step(f, np.ones(2, np.uint8))
    assert np.max(np.abs(eng.get_state() - P)) <= 1e-11 * np.max(np.abs(P))  # the suite's bar for states

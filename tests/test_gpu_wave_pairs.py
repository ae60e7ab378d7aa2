"""Odd band counts above 8 on grids whose k are stepped in stencil pairs: the last lane
of a k shares an element with the lane before it, and the second k of a pair reads its
accumulator late.  RK4 steps against the oracle's right-hand sides."""
import ctypes as C

import numpy as np
import pytest

from helpers import N, O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("diss", [False, True])
@pytest.mark.parametrize("nb", [9, 11, 15, 17, 19, 21, 23, 25, 27, 29, 31])
def test_rk4_of_odd_band_counts_on_a_paired_grid(nb, diss):
    rng = np.random.default_rng(nb + 100 * diss)
    n1, n2 = 3, 6
    nk, ncc, dp, ip = n1 * n2, nb // 2, C.POINTER(C.c_double), C.POINTER(C.c_int32)
    cplx = lambda *s: rng.normal(size=s) + 1j * rng.normal(size=s)  # noqa: E731
    H, P, U = cplx(nk, nb, nb), cplx(nk, nb, nb), np.linalg.qr(cplx(nk, nb, nb))[0]
    H, P = H + H.swapaxes(1, 2).conj(), P + P.swapaxes(1, 2).conj()
    D = rng.normal(size=(nk, nb, nb, 3)) + 0j
    D = D + D.swapaxes(1, 2)
    T = 0.1 * rng.uniform(size=(nb, nb)) if diss else np.zeros((nb, nb))
    i1, i2 = np.divmod(np.arange(nk), n2)
    off = [(0, 1), (0, -1), (1, 0), (-1, 0), (1, 1), (-1, -1)]
    nbr = np.stack([((i1 + a) % n1) * n2 + (i2 + b) % n2 for a, b in off], 1).astype(np.int32)
    wb, p, keep = rng.normal(size=(len(off), 3)), N.Problem(), []

    def host(a):
        keep.append(np.ascontiguousarray(a))
        return keep[-1].ctypes.data_as(dp)

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, 0, ncc, len(off), N.STEPPER_RK4, 4
    p.nbr, p.nbr_wb, p.H, p.D, p.U, p.T, p.rho0 = nbr.ctypes.data_as(ip), host(wb), host(H), host(D), host(U), host(T), host(P)
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.01, 1.0, 1.0, float(nk)
    eng, osys = N.Engine(p), O.System(H, D, U, T, nbr, np.ones(len(off)), wb, 0, ncc, 0.0)
    assert eng.launch_schedule()["stencil_pairs"] == 1
    f, dt = 0.3 * rng.normal(size=(3, 3, 6)), 0.01
    for E in f:
        k1 = osys.rhs(P, E[0], True)
        k2 = osys.rhs(P + dt / 2 * k1, E[1], True)
        k3 = osys.rhs(P + dt / 2 * k2, E[1], True)
        P = P + dt / 6 * (k1 + 2 * k2 + 2 * k3 + osys.rhs(P + dt * k3, E[2], True))
    eng.step(f, np.ones(len(f), np.uint8))
    assert np.max(np.abs(eng.get_state() - P)) <= 1e-11 * np.max(np.abs(P))  # the suite's bar for states

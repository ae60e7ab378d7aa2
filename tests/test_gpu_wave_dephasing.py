"""Dephasing of 5..32 bands on a grid's stencil: right-hand sides against the oracle
with and without rates of the filled bands (the hole source), grids that do and do
not pair, and a batch's member against the instance alone."""
import ctypes as C

import numpy as np
import pytest

from helpers import N, O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hole", [False, True])
@pytest.mark.parametrize("nb,n1,n2", [(5, 5, 7), (8, 6, 6), (9, 5, 7), (12, 6, 8), (16, 4, 6), (16, 3, 5), (17, 4, 6), (24, 3, 5), (32, 4, 4)])
def test_rhs_and_batch_with_dephasing(nb, n1, n2, hole):
    rng = np.random.default_rng(100 * nb + n1 + hole)
    nk, ncc, dp, ip = n1 * n2, nb // 2, C.POINTER(C.c_double), C.POINTER(C.c_int32)
    cplx = lambda *s: rng.normal(size=s) + 1j * rng.normal(size=s)  # noqa: E731
    H, P, U = cplx(nk, nb, nb), cplx(nk, nb, nb), np.linalg.qr(cplx(nk, nb, nb))[0]
    H, P = H + H.swapaxes(1, 2).conj(), P + P.swapaxes(1, 2).conj()
    D = rng.normal(size=(nk, nb, nb, 3)) + 0j
    D = D + D.swapaxes(1, 2)
    T = 0.1 * rng.uniform(size=(nb, nb))
    if not hole:
        T[range(ncc), range(ncc)] = 0.0
    i1, i2 = np.divmod(np.arange(nk), n2)
    nbr = np.stack([((i1 + a) % n1) * n2 + (i2 + b) % n2 for a, b in [(0, 1), (0, -1), (1, 0), (-1, 0)]], 1).astype(np.int32)
    wb, p, keep = rng.normal(size=(4, 3)), N.Problem(), []

    def host(a):
        keep.append(np.ascontiguousarray(a))
        return keep[-1].ctypes.data_as(dp)

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, 0, ncc, 4, N.STEPPER_RK4, 4
    p.nbr, p.nbr_wb, p.H, p.D, p.U, p.T, p.rho0 = nbr.ctypes.data_as(ip), host(wb), host(H), host(D), host(U), host(T), host(P)
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.01, 1.0, 1.0, float(nk)
    eng, osys = N.Engine(p), O.System(H, D, U, T, nbr, np.ones(4), wb, 0, ncc, 0.0)
    E = np.array([0.3, -0.2, 0.4, 0.1, 0.2, -0.3])
    for on in (True, False):
        got, ref = eng.rhs(E, on), osys.rhs(P, E, on)
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))  # the suite's bar for right-hand sides
    fields, on = 0.3 * rng.normal(size=(4, 3, 6)), np.ones(4, np.uint8)
    eng.step(fields, on)
    batch = N.Batch([p, p])
    batch.step([fields, fields], [on, on])
    for m in batch.members:
        assert np.array_equal(m.get_state(), eng.get_state())

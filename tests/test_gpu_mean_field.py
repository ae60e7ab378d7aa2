"""Right-hand side with the mean field for random tables against the oracle, where
the passes' tiles end: every band count they take, grids that are and are not
multiples of 16 or longer than one batch of the first pass, both bases, the screening
gate off and on."""
import ctypes as C

import numpy as np
import pytest

from helpers import N, O

pytestmark = pytest.mark.gpu


class _Coulomb(C.Structure):
    _fields_ = [("ncut", C.c_int32), ("diag_basis", C.c_int32)] + [(n, C.POINTER(C.c_double)) for n in ("A", "B", "C", "D", "screen", "vh")]


@pytest.mark.parametrize("nb,n1,n2,ncut,diag", [(1, 5, 7, 3, False), (2, 16, 16, 8, False), (3, 17, 33, 5, False), (4, 9, 40, 11, False),
                                                (2, 7, 5, 4, True), (3, 20, 17, 6, True), (4, 16, 18, 3, True), (2, 3, 200, 12, False),
                                                (1, 2, 385, 4, False)])
def test_rhs_with_mean_field_matches_oracle(nb, n1, n2, ncut, diag):
    rng = np.random.default_rng(10 * nb + n1)
    nk, ncc, dp, ip = n1 * n2, max(1, nb // 2), C.POINTER(C.c_double), C.POINTER(C.c_int32)
    cplx = lambda *s: rng.normal(size=s) + 1j * rng.normal(size=s)  # noqa: E731
    H = cplx(nk, nb, nb)
    H = H + H.swapaxes(1, 2).conj()
    D = rng.normal(size=(nk, nb, nb, 3)) + 0j
    D = D + D.swapaxes(1, 2)
    U = np.linalg.qr(cplx(nk, nb, nb))[0]
    rho0 = np.einsum("kvi,kvj->kij", U[:, :ncc], U[:, :ncc].conj())
    P = cplx(nk, nb, nb)
    P = 0.1 * (P + P.swapaxes(1, 2).conj()) + rho0
    off = [(0, 1), (0, -1), (1, 0), (-1, 0)]
    i1, i2 = np.divmod(np.arange(nk), n2)
    nbr = np.stack([((i1 + a) % n1) * n2 + (i2 + b) % n2 for a, b in off], 1).astype(np.int32)
    wb = rng.normal(size=(4, 3))
    cf = {q: 0.1 * cplx(ncut * ncut, nb * nb) for q in "ABCD"}
    for q in "AD":
        cf[q][:, 0] = cf[q][:, 0].real
    cf["screen"], cf["vh"] = cplx(nb * nb), rng.normal(size=(nb, nb)) + 0j
    p, q, keep = N.Problem(), _Coulomb(), []

    def host(a):
        keep.append(np.ascontiguousarray(a))
        return keep[-1].ctypes.data_as(dp)

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, 0, ncc, 4, N.STEPPER_RK4, 4
    p.nbr, p.nbr_wb, p.H, p.D, p.U, p.T, p.rho0 = nbr.ctypes.data_as(ip), host(wb), host(H), host(D), host(U), host(np.zeros((nb, nb))), host(rho0)
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.1, 1.0, 1.0, float(nk)
    p.nk_dims[0], p.nk_dims[1], p.nk_dims[2] = 1, n1, n2
    q.ncut, q.diag_basis = ncut, int(diag)
    for n in ("A", "B", "C", "D", "screen", "vh"):
        setattr(q, n, host(cf[n]))
    p.coulomb = C.cast(C.pointer(q), C.c_void_p)
    eng = N.Engine(p)
    osys = O.System(H, D, U, np.zeros((nb, nb)), nbr, np.ones(4), wb, 0, ncc, 0.0)
    osys.set_coulomb(ncut, O.kgrid(1, n1, n2), cf["A"], cf["B"], cf["C"], cf["D"], cf["screen"], cf["vh"], diag_basis=diag)
    E = np.array([0.1, -0.2, 0.3, 0.0, 0.0, 0.0])
    eng.set_state(P)
    for n_cond in (0.0, 1.0):
        got, ref = eng.rhs(E), osys.rhs_coulomb(rho0, P, E, True, n_cond)
        # the suite's bar for right-hand sides
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref)), n_cond
        eng.observables()  # the populations of this state open the gate

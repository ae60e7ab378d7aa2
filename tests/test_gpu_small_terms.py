"""The 1..4-band stage kernel, whose waves share out the terms of the right-hand
side: random tables against the oracle at every band count, with and without
dephasing, stencils that do not divide among the drift's waves and batches, grids
around the 64 k of a workgroup, and one step of each stepper."""
import ctypes as C

import numpy as np
import pytest

from helpers import N, O

pytestmark = pytest.mark.gpu


def _problem(nb, nk, nn, diss, nch, stepper, order, seed):
    rng = np.random.default_rng(seed)
    cplx = lambda *s: rng.normal(size=s) + 1j * rng.normal(size=s)  # noqa: E731
    t = {"H": cplx(nk, nb, nb), "D": cplx(nk, nb, nb, 3), "U": np.linalg.qr(cplx(nk, nb, nb))[0], "P": cplx(nk, nb, nb)}
    t["H"] = t["H"] + t["H"].swapaxes(1, 2).conj()
    t["P"] = t["P"] + t["P"].swapaxes(1, 2).conj()
    up = np.triu(t["D"].transpose(0, 3, 1, 2))
    idx = np.arange(nb)
    up[..., idx, idx] = up[..., idx, idx].real
    t["D"] = np.ascontiguousarray((up + np.triu(up, 1).swapaxes(2, 3)).transpose(0, 2, 3, 1))
    t["T"] = 0.1 * rng.uniform(size=(nb, nb)) if diss else np.zeros((nb, nb))
    t["nbr"] = rng.integers(0, nk, size=(nk, max(nn, 1))).astype(np.int32)[:, :nn].copy()
    t["wb"] = rng.normal(size=(max(nn, 1), 3))
    p, keep = N.Problem(), []

    def host(a):
        keep.append(np.ascontiguousarray(a))
        return keep[-1].ctypes.data_as(C.POINTER(C.c_double))

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, nch, max(1, nb // 2), nn, stepper, order
    p.nbr, p.nbr_wb = t["nbr"].ctypes.data_as(C.POINTER(C.c_int32)), host(t["wb"])
    p.H, p.D, p.U, p.T, p.rho0 = host(t["H"]), host(t["D"]), host(t["U"]), host(t["T"]), host(t["P"])
    p.dt, p.wx2, p.j_norm, p.tabs_norm, p.nktot = 0.01, 0.7 if nch else 0.0, 1.0, 1.0, 1.0
    if stepper == N.STEPPER_TAYLOR:
        tau = 0.01 * np.arange(1, order)
        p.taylor_tau_inv = host(np.linalg.inv(tau[:, None] ** np.arange(1, order)))
    t["keep"] = keep
    osys = O.System(t["H"], t["D"], t["U"], t["T"], t["nbr"] if nn else np.zeros((nk, 0), np.int32), np.ones(max(nn, 1)), t["wb"], nch,
                    max(1, nb // 2), p.wx2)
    return p, t, osys


@pytest.mark.parametrize("nb", [1, 2, 3, 4])
@pytest.mark.parametrize("nn,nk,diss,nch", [(0, 5, False, 0), (1, 63, True, 0), (5, 65, False, 1), (12, 64, True, 1), (13, 200, False, 0),
                                            (29, 129, True, 0), (64, 70, False, 0)])
def test_rhs_matches_oracle(nb, nn, nk, diss, nch):
    p, t, osys = _problem(nb, nk, nn, diss, min(nch, nb - 1), N.STEPPER_RK4, 4, 31 * nb + nn)
    eng = N.Engine(p)
    E = np.array([0.3, -0.2, 0.4, 0.1, 0.2, -0.3])
    for on in (1, 0):
        got, ref = eng.rhs(E, bool(on)), osys.rhs(t["P"], E, bool(on))
        assert np.max(np.abs(got - ref)) <= 1e-12 * max(np.max(np.abs(ref)), 1e-300)  # the suite's bar for right-hand sides


@pytest.mark.parametrize("nb,diss", [(1, False), (2, True), (3, False), (3, True), (4, False), (4, True)])
@pytest.mark.parametrize("stepper,order", [(N.STEPPER_RK4, 4), (N.STEPPER_AB, 2), (N.STEPPER_AB, 5), (N.STEPPER_TAYLOR, 2), (N.STEPPER_TAYLOR, 8)])
def test_steps_match_oracle_rhs(nb, diss, stepper, order):
    """Three steps put together from the oracle's right-hand sides."""
    p, t, osys = _problem(nb, 70, 12, diss, 0, stepper, order, 7 * nb + order)
    eng, dt, P, hist = N.Engine(p), 0.01, t["P"], []
    rng = np.random.default_rng(nb)
    f = 0.3 * rng.normal(size=(3, 3 if stepper == N.STEPPER_RK4 else 1, 6))
    eng.step(f, np.ones(3, np.uint8))
    ab = {2: [1.5, -0.5], 5: [1901 / 720, -2774 / 720, 2616 / 720, -1274 / 720, 251 / 720]}
    for E in f:
        k1 = osys.rhs(P, E[0])
        if stepper == N.STEPPER_RK4:
            k2 = osys.rhs(P + dt / 2 * k1, E[1])
            k3 = osys.rhs(P + dt / 2 * k2, E[1])
            P = P + dt / 6 * (k1 + 2 * k2 + 2 * k3 + osys.rhs(P + dt * k3, E[2]))
            continue
        h = (hist + [np.zeros_like(k1)] * order)[:order - 1]
        if stepper == N.STEPPER_AB:
            P = P + dt * sum(c * g for c, g in zip(ab[order], [k1] + h))
        else:
            ti = np.linalg.inv((dt * np.arange(1, order))[:, None] ** np.arange(1, order))
            P = P + dt * k1 + sum(dt ** (i + 1) / (i + 1) * sum(ti[i - 1, q] * (k1 - h[q]) for q in range(order - 1)) for i in range(1, order))
        hist = ([k1] + hist)[:order - 1]
    # the suite's bar for states, times the size of tau^-1 that Taylor's differences are multiplied with
    bar = 1e-11 * (1.0 if stepper != N.STEPPER_TAYLOR else max(1.0, np.max(np.abs(ti * dt ** np.arange(1, order)[:, None]))))
    assert np.max(np.abs(eng.get_state() - P)) <= bar * np.max(np.abs(P))

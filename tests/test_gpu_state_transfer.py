"""States of both layouts to the caller's full matrices, by the host's loop and, from
16 MB on, unpacked on the device: one piece, a last piece of a few k, odd counts.
A transfer does not wait for other contexts."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from helpers import N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nk", [(1, 7), (3, 1001), (4, 65535), (4, 65536), (3, 466033 + 5), (5, 50001), (16, 4097), (17, 14513), (32, 1024),
                                   (32, 4099)])
def test_state_round_trip(nb, nk):
    rng = np.random.default_rng(nb)
    P = rng.normal(size=(nk, nb, nb)) + 1j * rng.normal(size=(nk, nb, nb))
    P += P.swapaxes(1, 2).conj()
    dp = C.POINTER(C.c_double)
    unit, zero = np.broadcast_to(np.eye(nb) + 0j, (nk, nb, nb)).copy(), np.zeros((nk, nb, nb, 3), complex)
    T, w = np.zeros((nb, nb)), np.zeros((1, 3))
    p = N.Problem()
    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, 0, 1, 0, N.STEPPER_RK4, 4
    nbr = np.zeros((nk, 1), np.int32)
    p.nbr, p.nbr_wb = nbr.ctypes.data_as(C.POINTER(C.c_int32)), w.ctypes.data_as(dp)
    p.H, p.D, p.U, p.T, p.rho0 = (a.ctypes.data_as(dp) for a in (unit, zero, unit, T, P))
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.01, 1.0, 1.0, float(nk)
    eng = N.Engine(p)
    assert np.array_equal(eng.get_state(), P)
    eng.set_state(P[::-1])
    assert np.array_equal(eng.get_state(), P[::-1])


def _engine(P):
    nk, nb = P.shape[:2]
    dp = C.POINTER(C.c_double)
    unit, zero = np.broadcast_to(np.eye(nb) + 0j, (nk, nb, nb)).copy(), np.zeros((nk, nb, nb, 3), complex)
    T, w = np.zeros((nb, nb)), np.zeros((1, 3))
    p = N.Problem()
    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, 0, 1, 0, N.STEPPER_RK4, 4
    nbr = np.zeros((nk, 1), np.int32)
    p.nbr, p.nbr_wb = nbr.ctypes.data_as(C.POINTER(C.c_int32)), w.ctypes.data_as(dp)
    p.H, p.D, p.U, p.T, p.rho0 = (a.ctypes.data_as(dp) for a in (unit, zero, unit, T, P))
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.01, 1.0, 1.0, float(nk)
    return N.Engine(p)


def test_transfer_does_not_wait_for_another_context():
    """An 82 MB state while another context's steps are queued: in well under their time,
    of the first transfer too (that allocates what the context keeps for the later ones)."""
    P = np.ones((80000, 8, 8), complex)
    mine, fresh, other = _engine(P), _engine(P), _engine(np.ones((16384, 32, 32), complex))
    mine.get_state()
    n = 400
    steps = threading.Thread(target=other.step, args=(np.zeros((n, 3, 6)), np.ones(n, np.uint8)))
    steps.start()
    time.sleep(0.02)  # the launches are queued meanwhile
    took = []
    for e in (mine, fresh, mine):
        t = time.perf_counter()
        state = e.get_state()
        took.append(1e3 * (time.perf_counter() - t))
        assert np.array_equal(state, P)
    steps.join()
    ms = other.last_step_time()[0]
    assert ms > 80 and max(took) < 0.4 * ms, (took, ms)

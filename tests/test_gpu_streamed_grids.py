"""1..4 bands on grids whose arrays exceed the caches, where the stage kernel reads its
operands as streams: a problem repeated until it is that large steps every copy to the
bits of the small problem."""
import ctypes as C

import numpy as np
import pytest

from helpers import N
from test_gpu_small_terms import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,diss,stepper,order", [(1, True, N.STEPPER_RK4, 4), (2, False, N.STEPPER_AB, 4), (3, False, N.STEPPER_RK4, 4),
                                                   (3, True, N.STEPPER_TAYLOR, 3), (4, True, N.STEPPER_AB, 3), (4, False, N.STEPPER_RK4, 4)])
def test_repeated_problem_steps_like_one(nb, diss, stepper, order):
    nk, nn = 10007, 12
    p, t, _ = _problem(nb, nk, nn, diss, 0, stepper, order, nb)
    m = int(360e6 / (nk * (4 * nn + 48 * nb * nb))) + 1
    fields, on = 0.3 * np.random.default_rng(nb).normal(size=(3, 3 if stepper == N.STEPPER_RK4 else 1, 6)), np.ones(3, np.uint8)
    one = N.Engine(p)
    one.step(fields, on)
    big, keep = N.Problem(), []
    for f, _ in N.Problem._fields_:
        setattr(big, f, getattr(p, f))
    big.nk = m * nk
    for f, a in (("H", t["H"]), ("D", t["D"]), ("U", t["U"]), ("rho0", t["P"])):
        keep.append(np.tile(a, (m,) + (1,) * (a.ndim - 1)))
        setattr(big, f, keep[-1].ctypes.data_as(C.POINTER(C.c_double)))
    nbr = (t["nbr"][None] + nk * np.arange(m, dtype=np.int32)[:, None, None]).reshape(-1, nn)
    big.nbr = nbr.ctypes.data_as(C.POINTER(C.c_int32))
    eng = N.Engine(big)
    eng.step(fields, on)
    want, got = one.get_state(), eng.get_state().reshape(m, nk, nb, nb)
    assert np.isfinite(want).all() and not np.array_equal(want, t["P"])
    for i in range(m):
        assert np.array_equal(got[i], want), i

"""Sums of the observables over the grid that cancel: large terms of opposite signs at
scattered k, small ones in between.  One matrix element is filled, every product is
exact, so what is left of the small terms shows whether each addition over k kept its
rounding error, in every band class and on both sides of the kernels' block sizes."""
import ctypes as C

import numpy as np
import pytest

from helpers import N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("diag", [True, False])
@pytest.mark.parametrize("nb,nk", [(1, 300), (2, 64), (3, 1001), (4, 70000), (5, 13), (7, 9001), (8, 20000), (9, 5), (13, 3100), (16, 700), (17, 800),
                                   (24, 1600), (32, 1600)])
def test_sums_over_k_keep_their_rounding_errors(nb, nk, diag):
    if nb == 1 and not diag:
        pytest.skip("one band has no off-diagonal element")
    rng = np.random.default_rng(1000 * nb + nk)
    third = nk // 3
    big = (rng.integers(2 ** 20, 2 ** 22, size=third) * 2 + 1) * 2.0 ** 30
    small = rng.integers(1, 1000, size=nk - 2 * third).astype(float)
    v = rng.permutation(np.concatenate([big, -big, small]))  # its sum is that of `small`
    i, j = 0, 0 if diag else nb - 1
    P = np.zeros((nk, nb, nb), dtype=np.complex128)
    z = 1.0 if diag else 1.0 + 2.0j
    P[:, i, j] = v * z
    P[:, j, i] = v * np.conj(z)
    gx, dx = np.array([1.0, 2.0, -4.0]), np.array([0.5, -1.0, 2.0])
    G, D = np.zeros((2, nk, nb, nb, 3), dtype=np.complex128)
    G[:, i, j] = G[:, j, i] = gx
    D[:, i, j] = D[:, j, i] = dx
    one = np.broadcast_to(np.eye(nb, dtype=np.complex128), (nk, nb, nb)).copy()
    nch = 0 if diag else 1
    p, keep = N.Problem(), []

    def host(a):
        keep.append(np.ascontiguousarray(a))
        return keep[-1].ctypes.data_as(C.POINTER(C.c_double))

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, nch, max(nch, 1), 0, N.STEPPER_RK4, 4
    p.nbr, p.nbr_wb = np.zeros(1, dtype=np.int32).ctypes.data_as(C.POINTER(C.c_int32)), host(np.zeros(3))
    p.H, p.U, p.D, p.gradH, p.T, p.rho0 = host(one), host(one), host(D), host(G), host(np.zeros((nb, nb))), host(P)
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.1, 1.0, 1.0, 1.0
    got = N.Engine(p).observables()
    total, moduli, u = small.sum(), np.abs(v).sum(), 2.0 ** -53
    # Sums with kept errors (Sum2 of Ogita, Rump and Oishi 2005): u |S| + gamma^2 sum |x|,
    # nk additions that are not exact; the factors of the elements are powers of two
    tol = 2 * u * total + (nk * u) ** 2 * moduli
    pairs = 1 if diag else 2  # an off-diagonal element and its mirror
    assert np.all(np.abs(got["j1"][0::2] - pairs * gx * total) <= pairs * np.abs(gx) * tol)
    assert np.all(np.abs(got["j2"][0::2] - pairs * dx * total) <= pairs * np.abs(dx) * tol)
    if diag:
        assert abs(got["pop"][0] - total) <= tol and not got["pop"][1:].any() and not got["tabs"].any()
    else:
        ta = -2 * dx * total
        assert np.all(np.abs(got["tabs"][0::2] - ta) <= np.abs(ta) / total * tol)
        assert np.all(np.abs(got["tabs"][1::2] - 2 * ta) <= 2 * np.abs(ta) / total * tol)

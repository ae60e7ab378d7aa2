"""Observables and snapshot elements of random Hermitian states against numpy, at
the edges of their kernels: every band class, odd band counts, one k, remainders
of the blocks' k, more k than one round of blocks, symmetric and Hermitian dipoles.
"""
import ctypes as C

import numpy as np
import pytest

from helpers import N

pytestmark = pytest.mark.gpu


def _hermitian(rng, nk, nb, n=None):
    a = rng.normal(size=(nk, nb, nb) + ((n,) if n else ())) + 1j * rng.normal(size=(nk, nb, nb) + ((n,) if n else ()))
    return a + np.swapaxes(a, 1, 2).conj()


def _engine(nk, nb, nch, ncc, herm, seed, gradient=True):
    rng = np.random.default_rng(seed)
    H, G, D = _hermitian(rng, nk, nb), _hermitian(rng, nk, nb, 3), _hermitian(rng, nk, nb, 3)
    if not herm:  # symmetric with a real diagonal
        up = np.triu(D.transpose(0, 3, 1, 2))
        D = (up + np.triu(up, 1).swapaxes(2, 3)).transpose(0, 2, 3, 1)
    U = np.linalg.qr(rng.normal(size=(nk, nb, nb)) + 1j * rng.normal(size=(nk, nb, nb)))[0]
    P = _hermitian(rng, nk, nb)
    p, keep = N.Problem(), []

    def host(a):
        keep.append(np.ascontiguousarray(a))
        return keep[-1].ctypes.data_as(C.POINTER(C.c_double))

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr, p.stepper, p.order = nk, nb, nch, ncc, 0, N.STEPPER_RK4, 4
    p.nbr, p.nbr_wb = np.zeros(1, dtype=np.int32).ctypes.data_as(C.POINTER(C.c_int32)), host(np.zeros(3))
    p.H, p.D, p.U, p.T, p.rho0 = host(H), host(D), host(U), host(np.zeros((nb, nb))), host(P)
    if gradient:
        p.gradH = host(G)
    p.dt, p.j_norm, p.tabs_norm, p.nktot = 0.1, 1.0, 1.0, 1.0
    return N.Engine(p), H, D, U, G, P


@pytest.mark.parametrize("nb,nk,nch,ncc,herm", [
    (1, 3, 0, 1, False), (2, 257, 1, 1, True), (3, 256, 1, 2, False), (4, 1001, 0, 2, True),
    (5, 13, 1, 2, False), (7, 8200, 0, 3, True), (8, 8193, 2, 4, False),
    (9, 1, 1, 4, True), (13, 3083, 0, 6, False), (16, 3074, 3, 8, True),
    (17, 2, 0, 8, False), (24, 769, 2, 12, True), (32, 1537, 0, 16, False)])
def test_observables_and_elements_match_numpy(nb, nk, nch, ncc, herm):
    eng, H, D, U, G, P = _engine(nk, nb, nch, ncc, herm, 100 * nb + nk)
    got = eng.observables()
    # every value is a sum of products of at most three factors through inner sums
    # of nb terms: a first-order bound of (4 nb + 64) half-ulps of the sum of moduli
    eps = (4 * nb + 64) * 2.0 ** -53
    aP, aU, aD = np.abs(P), np.abs(U), np.abs(D)
    pk = np.einsum("kci,kij,kcj->kc", U.conj(), P, U, optimize=True).real
    bound = np.einsum("kci,kij,kcj->kc", aU, aP, aU, optimize=True)
    assert np.all(np.abs(got["pop"] - pk.sum(0)) <= eps * bound.sum(0))
    hole = np.where(np.arange(nb) < ncc, 1 - pk, pk)
    tol = eps * (1 + bound.max())
    assert abs(got["pminmax"][0] - min(1.0, hole.min())) <= tol and abs(got["pminmax"][1] - np.abs(hole).max()) <= tol
    j1 = np.einsum("kij,kijx->x", P, G)
    assert np.all(np.abs(got["j1"][0::2] - j1.real) <= eps * np.einsum("kij,kijx->x", aP, np.abs(G))) and not got["j1"][1::2].any()
    j2 = np.einsum("kij,kic,kjcx->x", P, H, D.conj(), optimize=True)
    b2 = np.einsum("kij,kic,kjcx->x", aP, np.abs(H), aD, optimize=True)
    assert np.all(np.abs(got["j2"][0::2] + 1j * got["j2"][1::2] - j2) <= eps * b2)
    ta = -2 * np.einsum("kij,kijx->x", P[:, :nch, nch:], D[:, :nch, nch:])
    bt = 2 * np.einsum("kij,kijx->x", aP[:, :nch, nch:], aD[:, :nch, nch:])
    assert np.all(np.abs(got["tabs"][0::2] + 1j * got["tabs"][1::2] - ta) <= eps * bt)
    again = eng.observables()  # the arrival counter is back at zero; the sums' order is fixed
    assert all(np.array_equal(got[k], again[k]) for k in got)
    for i, j in {(0, 0), (nb - 1, 0), (0, nb - 1), (nb // 2, nb - 1)}:
        v = np.einsum("ki,kij,kj->k", U[:, i].conj(), P, U[:, j])
        v = v.real + 0j if i == j else v
        assert np.all(np.abs(eng.eigen_element(i, j) - v) <= eps * np.einsum("ki,kij,kj->k", aU[:, i], aP, aU[:, j]))


@pytest.mark.parametrize("nb", [3, 12])
def test_no_gradient_table_gives_no_first_current(nb):
    eng = _engine(70, nb, 0, 1, True, 7, gradient=False)[0]
    assert not eng.observables()["j1"].any()


def test_contexts_beyond_one_slab_of_results():
    """Result slots of many contexts at once, freed and taken again."""
    engs = [_engine(5, 2, 0, 1, True, i) for i in range(70)]
    want = [np.einsum("kci,kij,kcj->c", e[3].conj(), e[5], e[3]).real for e in engs]
    for r in range(2):
        for e, w in zip(engs[::-1], want[::-1]):
            assert np.allclose(e[0].observables()["pop"], w, rtol=0, atol=1e-12)
        for e in engs[:65]:
            e[0].close()
        engs, want = engs[65:], want[65:]

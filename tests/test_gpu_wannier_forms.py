"""Wannier contraction against a direct sum where its kernels and copies branch: band
counts around the 64-column tiles, grids that are no multiple of 64 k, one lattice
vector and lists that do not fill a tile of 16, H(R) and r(R) without symmetry,
results large enough for the threaded download."""
import numpy as np
import pytest

from helpers import N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,nk3,nR", [(1, (1, 3, 5), 1), (2, (1, 8, 8), 17), (5, (2, 7, 9), 16), (7, (1, 13, 5), 33), (9, (1, 65, 1), 5),
                                       (17, (1, 6, 11), 20), (32, (1, 9, 9), 7), (8, (1, 181, 200), 6)])
@pytest.mark.parametrize("form", ["fp64", "fp32", "bf16x3"])
def test_contraction_matches_direct_sum(nw, nk3, nR, form):
    rng = np.random.default_rng(nw + nR)
    R = rng.integers(-6, 7, size=(nR, 3)).astype(np.int32)
    HR = rng.normal(size=(nR, nw, nw)) + 1j * rng.normal(size=(nR, nw, nw))
    rR = rng.normal(size=(nR, nw, nw, 3)) + 1j * rng.normal(size=(nR, nw, nw, 3))
    ax = [(-0.5 + np.arange(n) / n) if n > 1 else np.zeros(1) for n in nk3]
    k = np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    ph = np.exp(2j * np.pi * (k @ R.T))
    H = (ph @ HR.reshape(nR, -1)).reshape(-1, nw, nw)
    D = (ph @ rR.reshape(nR, -1)).reshape(-1, nw, nw, 3)
    i = np.arange(nw)
    H[:, i, i] = H[:, i, i].real
    D[:, i, i] = D[:, i, i].real
    D = 0.5 * (D + D.swapaxes(1, 2))
    h, d = N.wannier_hk(list(nk3), R, HR, rR, nw, fp32=form == "fp32", bf16x3=form == "bf16x3")
    # the bounds that include/edus.h states for the forms; FP64 with its own unit
    # roundoff, the phases' and the reference sum's
    per = {"fp64": (4 * nR + 40) * 2.0 ** -53, "fp32": (2 * nR + 4) * 2.0 ** -24,
           "bf16x3": np.sqrt(2) * (3 * 2.0 ** -18 + (2 * nR + 8) * 2.0 ** -24)}[form]
    sr = np.abs(rR).sum(0)
    assert np.all(np.abs(h - H) <= per * np.abs(HR).sum(0))
    assert np.all(np.abs(d - D) <= per * 0.5 * (sr + sr.swapaxes(0, 1)) * (1 + 1e-6))
    if form == "fp64":
        assert np.array_equal(h[:, i, i].imag, np.zeros((len(k), nw))) and np.array_equal(d, d.swapaxes(1, 2))

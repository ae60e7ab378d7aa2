"""Coulomb coefficient generator against the oracle where its kernels branch: every
band count, both potentials, lists of G that are and are not closed under G -> -G,
shorter and longer than a tile, an even Simpson grid, more Fourier modes than the
correction's table holds, a correction grid without points."""
import numpy as np
import pytest

from helpers import N, O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,ry,ncut,n_sum,n_peak,shell,cut", [
    (1, 1, 3, 21, 401, 3, 0), (2, 0, 17, 31, 401, 6, 0), (3, 1, 5, 32, 801, 8, 1), (4, 1, 20, 41, 401, 7, 0), (4, 0, 2, 25, 3, 5, 7),
    (2, 1, 25, 61, 801, 12, 3)])
def test_generator_matches_oracle(nb, ry, ncut, n_sum, n_peak, shell, cut):
    rng = np.random.default_rng(nb + n_sum)
    m = np.arange(-shell, shell + 1)
    g = np.stack(np.meshgrid(m, m, indexing="ij"), -1).reshape(-1, 2)
    g = g[(g ** 2).sum(1) < shell * shell]
    g = g[cut:]  # cut > 0: the list loses its mirror symmetry
    disp = np.zeros((nb, 3))
    disp[:, 1:] = rng.uniform(-1.5, 1.5, size=(nb, 2))
    p = {"nb": nb, "ncut": ncut, "n_sum": n_sum, "n_peak": n_peak, "rytova": ry, "g": g, "b1": np.array([0.0, 1.4, 0.3]),
         "b2": np.array([0.1, -0.5, 1.2]), "eps_area": 19.3, "qtf": 0.05, "r0": 18.9, "q_peak": 0.05, "disp": disp}
    gpu, ora = N.coulomb_coefficients(p), O.coulomb_coefficients(p)
    for k in ("A", "B", "C", "D", "vh", "screen"):  # the suite's bars for the generator
        assert np.max(np.abs(gpu[k] - ora[k])) <= (1e-10 if k == "screen" else 1e-11) * max(np.max(np.abs(ora[k])), 1e-300), k
    again = N.coulomb_coefficients(p)
    assert all(np.array_equal(gpu[k], again[k]) for k in gpu)


def test_unscreened_potential_at_the_origin_is_infinite():
    """qTF = 0 on a grid that holds q = 0: V(0) = 2 pi / 0, as the formula gives it."""
    p = {"nb": 1, "ncut": 1, "n_sum": 5, "n_peak": 3, "rytova": 1, "g": np.array([[0, 0]]), "b1": np.array([0.0, 1.0, 0.0]),
         "b2": np.array([0.0, 0.0, 1.0]), "eps_area": 1.0, "qtf": 0.0, "r0": 1.0, "q_peak": 0.0, "disp": np.zeros((1, 3))}
    assert np.isposinf(N.coulomb_coefficients(p)["A"][0, 0].real)


@pytest.mark.parametrize("ry,qtf,r0", [(1, 0.05, -1000.0), (1, 0.05, 1e160), (1, 1e160, 1e150), (0, 1e160, 1.0), (1, 1e-160, 18.9),
                                       (1, 0.05, 0.0)])
def test_generator_with_extreme_screening_matches_oracle(ry, qtf, r0):
    """Parameters for which (q^2 + qTF^2) (|q| r0 + 1)^2 overflows, is not a normal number
    or loses the sign of |q| r0 + 1 (no q of these grids is near its zero)."""
    m = np.arange(-4, 5)
    g = np.stack(np.meshgrid(m, m, indexing="ij"), -1).reshape(-1, 2)
    p = {"nb": 2, "ncut": 3, "n_sum": 20, "n_peak": 400, "rytova": ry, "g": g, "b1": np.array([0.0, 1.4, 0.3]),
         "b2": np.array([0.1, -0.5, 1.2]), "eps_area": 19.3, "qtf": qtf, "r0": r0, "q_peak": 0.05, "disp": np.array([[0.0, 0.3, 0.1], [0.0, -0.7, 1.0]])}
    gpu, ora = N.coulomb_coefficients(p), O.coulomb_coefficients(p)
    for k in ("A", "B", "C", "D", "vh", "screen"):
        assert np.all(np.isfinite(ora[k])), k
        assert np.max(np.abs(gpu[k] - ora[k])) <= (1e-10 if k == "screen" else 1e-11) * max(np.max(np.abs(ora[k])), 1e-300), k

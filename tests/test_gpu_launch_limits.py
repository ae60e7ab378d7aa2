"""Calls at the ends of their launch rules: more Fourier modes than one load block of
the mean field's passes (20 of k_coul_w_mfma, 10 of k_coul_s3) up to the 32 that are
accepted, and the workgroup sizes that edus_autotune launches at 1..4 bands, among them
128 k of 4 bands with dephasing, whose terms fill the 64 KB of LDS (the size it keeps,
checked here, is a matter of timing)."""
import numpy as np
import pytest

import test_gpu_mean_field as mean_field
from helpers import N
from test_gpu_small_terms import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,n1,n2,ncut,diag", [(3, 17, 20, 21, False), (2, 8, 33, 31, False), (4, 18, 7, 32, False), (1, 6, 40, 32, True), (3, 16, 9, 25, True)])
def test_mean_field_with_many_modes(nb, n1, n2, ncut, diag):
    mean_field.test_rhs_with_mean_field_matches_oracle(nb, n1, n2, ncut, diag)


@pytest.mark.parametrize("nb,diss", [(1, False), (2, True), (3, True), (4, False), (4, True)])
def test_workgroup_sizes_of_the_small_kernel(nb, diss):
    p, t, osys = _problem(nb, 1003, 6, diss, 1, N.STEPPER_RK4, 4, 10 * nb + diss)
    eng = N.Engine(p)
    E = 0.3 * np.random.default_rng(nb).normal(size=6)
    ref, seen = osys.rhs(t["P"], E, True), set()
    for _ in range(12):  # the timing of a single launch falls one way and the other
        seen.add(eng.autotune(E, True, reps=1))
        assert np.max(np.abs(eng.rhs(E) - ref)) <= 1e-12 * np.max(np.abs(ref))  # the suite's bar for right-hand sides
    print("k per workgroup:", sorted(seen), flush=True)
    assert seen <= ({64, 128, 256} if nb <= 2 and not diss else {64, 128})

"""The signs of RHF's orbitals do not depend on those LAPACK gives."""
import numpy as np

from nopt_amd.scf import fix_signs


def test_signs_are_fixed():
    rng = np.random.default_rng(2)
    C = rng.standard_normal((7, 5))
    C[3, 2], C[5, 2] = 9.0, -9.0 * (1.0 + 1e-9)  # equal by symmetry but for rounding: the first decides
    want = fix_signs(C)
    assert want[3, 2] == 9.0
    assert np.array_equal(np.abs(want), np.abs(C))
    for signs in ([1, -1, 1, -1, 1], [-1, -1, -1, -1, -1]):
        assert np.array_equal(fix_signs(C * np.array(signs)), want)

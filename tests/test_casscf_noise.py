"""CASSCF with builds that round as coarsely as the integer mode: the energy is
then uneven by 1e-6 Eh while the gradient still tells the way. J and K from B,
the orbitals and the half-transform rounded to 24 bits below each row's largest
value (a relative error of 2e-8 in K; the integer mode has 3e-8). CPU only."""
import numpy as np
import pytest

from nopt_amd.casscf import CASSCF
from nopt_amd.molecule import Molecule
from nopt_amd.scf import rhf
from systems import SYSTEMS, CAS_C2H4
from test_casscf import _NumpyJK


def rounded(a, bits=24):
    mx = np.abs(a).max(axis=-1, keepdims=True)
    s = 2.0 ** (bits - np.ceil(np.log2(np.where(mx > 0.0, mx, 1.0))))
    return np.rint(a * s) / s


@pytest.fixture(scope="module")
def c2h4():
    sym, xyz = SYSTEMS["C2H4"]
    m = Molecule.from_angstrom(sym, xyz, basis="cc-pvdz", aux="cc-pvdz-ri")
    host = _NumpyJK(m)
    Br = rounded(host.B)

    def coarse(items):
        out = []
        for D, C, n in items:
            X = rounded(Br @ rounded(np.asarray(C)[:n]).T)
            out.append((host.build(D, C, 0)[0], np.tensordot(X, X, axes=([0, 2], [0, 2]))))
        return out
    return m, host, coarse, rhf(m, ctx=host, e_conv=1e-12, d_conv=1e-10).C


@pytest.mark.parametrize("seed", range(6))
def test_coarse_builds_reach_their_threshold(c2h4, seed):
    """From RHF orbitals turned by 1e-3 at random: a gradient of 1e-4 within 30
    steps, from where the exact builds finish."""
    m, host, coarse, C = c2h4
    rng = np.random.default_rng(seed)
    k = 1e-3 * rng.standard_normal((C.shape[1],) * 2)
    C0 = C @ np.linalg.qr(np.eye(len(k)) + k - k.T)[0]
    args = dict(n_core=m.nocc - 1, n_act=2, n_alpha=1, n_beta=1, nstates=2, mult=1)
    out = CASSCF(m, coarse, host.Bp, **args).run(C0, g_conv=1e-4, e_conv=1e-7, max_it=30)
    print("coarse", out["converged"], out["iters"], out["gmax"], out["E"] - CAS_C2H4["E_avg"])
    assert out["converged"] and out["gmax"] < 1e-4
    assert abs(out["E"] - CAS_C2H4["E_avg"]) < 2e-6
    end = CASSCF(m, host.build_batch, host.Bp, **args).run(out["C"])
    print("exact", end["converged"], end["iters"], end["E"] - CAS_C2H4["E_avg"])
    assert end["converged"] and abs(end["E"] - CAS_C2H4["E_avg"]) < 1e-9

"""The integer-build CASSCF of C2H4, refined in FP64 builds, from RHF orbitals
of any signs and slightly turned: the integer stage's rounding depends on them,
and where it stops must not."""
import numpy as np
import pytest

from nopt_amd.casscf import CASSCF, gpu_jk
from nopt_amd.jk import JKContext
from nopt_amd.molecule import Molecule
from nopt_amd.scf import rhf
from systems import SYSTEMS, CAS_C2H4

pytestmark = pytest.mark.gpu


def test_integer_builds_reach_their_threshold_from_any_signs():
    sym, xyz = SYSTEMS["C2H4"]
    m = Molecule.from_angstrom(sym, xyz, basis="cc-pvdz", aux="cc-pvdz-ri")
    args = dict(n_core=m.nocc - 1, n_act=2, n_alpha=1, n_beta=1, nstates=2, mult=1)
    with JKContext(m.nbf, m.naux) as ctx:
        ctx.set_B(m.eri3_packed(), m.metric())
        C = rhf(m, ctx=ctx, e_conv=1e-12, d_conv=1e-10).C
        B = ctx.get_B()
        for seed in range(16):
            rng = np.random.default_rng(seed)
            C0 = C * rng.choice([-1.0, 1.0], C.shape[1])
            if seed >= 8:
                k = 1e-6 * rng.standard_normal((C.shape[1],) * 2)
                C0 = C0 @ np.linalg.qr(np.eye(len(k)) + k - k.T)[0]
            i8 = CASSCF(m, gpu_jk(ctx, "int8"), B, **args).run(C0, g_conv=1e-4, e_conv=1e-7, max_it=60)
            print("seed", seed, "int8", i8["converged"], i8["iters"], i8["gmax"], i8["E"] - CAS_C2H4["E_avg"], flush=True)
            assert i8["converged"] and abs(i8["E"] - CAS_C2H4["E_avg"]) < 2e-6
            f64 = CASSCF(m, gpu_jk(ctx, "fp64"), B, **args).run(i8["C"])
            print("  fp64", f64["converged"], f64["iters"], f64["E"] - CAS_C2H4["E_avg"], flush=True)
            assert f64["converged"] and abs(f64["E"] - CAS_C2H4["E_avg"]) < 1e-9

"""B = L^-1 (P|mn) for metrics whose 64 x 64 diagonal blocks are as ill
conditioned as those of fitting bases. L has entries of -1, 0 and 1 and a unit
diagonal, so V = L L^T, its factorisation and the inverses of the factor's
diagonal blocks are whole numbers and exact, while those inverses grow to 1e6
and beyond; T = L B0 with B0 of order one cancels in the products with them. What
is left is the substitution's own error, held to the bound of a substitution in
rows and blocks: each row of L B misses T by the roundings of at most n + 64
products and sums of |L| |B| (once for the sums, once for the refined block)."""
import numpy as np
import pytest

from nopt_amd.jk import JKContext
from test_gpu_fp64 import say

pytestmark = pytest.mark.gpu


def factor(n, seed=5):
    rng = np.random.default_rng(seed)
    L = np.tril(rng.integers(-1, 2, (n, n)).astype(np.float64), -1)
    return L + np.eye(n)


def block_conditions(L):
    return [np.linalg.cond(L[k:k + 64, k:k + 64]) for k in range(0, len(L), 64)]


def excess(L, B, T):
    """Largest |L B - T| / bound, evaluated in extended precision."""
    n = len(L)
    worst = 0.0
    for s in range(0, T.shape[1], 4096):
        Lx, Bx = L.astype(np.longdouble), B[:, s:s + 4096].astype(np.longdouble)
        r = np.abs(Lx @ Bx - T[:, s:s + 4096]).astype(np.float64)
        bound = 2.0 * (n + 64) * 2.0 ** -53 * (np.abs(L) @ np.abs(B[:, s:s + 4096]))
        worst = max(worst, float((r / bound).max()))
    return worst


# the last one: 32896 columns, so that the 130 functions arrive in three groups
# of 64 and less, the later ones solved against the rows before them, and 34 MB,
# which go through the pinned pieces
@pytest.mark.parametrize("naux,nbf", [(63, 8), (64, 20), (130, 24), (200, 9), (130, 256)])
def test_substitution_through_ill_conditioned_blocks(naux, nbf):
    L = factor(naux)
    V = L @ L.T
    rng = np.random.default_rng(9)
    T = L @ rng.standard_normal((naux, nbf * (nbf + 1) // 2))
    say("naux", naux, "nbf", nbf, "conditions", ["%.1e" % c for c in block_conditions(L)])
    with JKContext(nbf, naux, keep="fp64") as ctx:
        ctx.set_B(T, V)
        B = ctx.get_B()
    worst = excess(L, B, T)
    say("  max residual / bound", worst)
    assert worst <= 1.0

"""The FP64 contraction kernels at the edges of their tiles, against numpy in
FP64: J and K of random B, D and C through the C-ABI. Every element is held to
the forward error bound of the nested sums, N u times the same sums over
absolute values with N the number of terms that are added (twice, for numpy's
own rounding), in any order of the sums."""
import sys

import numpy as np
import pytest

from nopt_amd.jk import JKContext

pytestmark = pytest.mark.gpu

# rows: 64-row tiles and 16-row blocks of the exchange, one and several; columns: 4, 16, one and several column groups
SHAPES = [(1, 1, 1), (2, 5, 2), (15, 3, 4), (16, 9, 5), (17, 9, 16), (24, 116, 5), (63, 7, 17), (64, 7, 20),
          (65, 7, 63), (80, 13, 80), (129, 21, 81), (144, 6, 129), (200, 11, 136), (210, 4, 210)]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def jk(B, D, C):
    X = np.einsum("qmn,in->qmi", B, C, optimize=True)
    return np.einsum("qmn,q->mn", B, np.einsum("qmn,mn->q", B, D, optimize=True), optimize=True), \
        np.einsum("qmi,qni->mn", X, X, optimize=True)


def inputs(nbf, naux, nocc, seed=3):
    rng = np.random.default_rng(seed)
    B = rng.standard_normal((naux, nbf, nbf))
    B = 0.5 * (B + B.transpose(0, 2, 1))
    C = rng.standard_normal((nocc, nbf))
    D = rng.standard_normal((nbf, nbf))
    r, c = np.tril_indices(nbf)
    return B, np.ascontiguousarray(B[:, r, c]), 0.5 * (D + D.T), C


def check(got, want, bound, terms):
    tol = 2.0 * terms * 2.0 ** -53 * bound
    say("  max error / bound", float(np.max(np.abs(got - want) / tol)))
    assert np.all(np.abs(got - want) <= tol)
    assert np.array_equal(got, got.T)


@pytest.mark.parametrize("nbf,naux,nocc", SHAPES)
def test_fp64_build_at_tile_edges(nbf, naux, nocc):
    say("nbf", nbf, "naux", naux, "nocc", nocc)
    B, packed, D, C = inputs(nbf, naux, nocc)
    J0, K0 = jk(B, D, C)
    Ja, Ka = jk(np.abs(B), np.abs(D), np.abs(C))
    with JKContext(nbf, naux, keep="fp64") as ctx:
        ctx.set_B_fitted(packed)
        J, K = ctx.build(D, C, prec="fp64")
        check(J, J0, Ja, nbf * nbf + naux + 2)
        check(K, K0, Ka, 2 * nbf + naux * nocc + 2)
        J2, K2 = ctx.build(D, C, prec="fp64")
        assert np.array_equal(J, J2) and np.array_equal(K, K2)
        assert np.array_equal(ctx.build(None, C, prec="fp64", J=False)[1], K)


@pytest.mark.parametrize("nbf,naux,na", [(1, 1, 1), (16, 31, 4), (17, 33, 16), (63, 32, 17), (64, 5, 8), (130, 40, 32)])
def test_active_integrals_at_tile_edges(nbf, naux, na):
    """Two different orbital sets: ints = sum_Q R_Q R_Q, R_Q = C2 B_Q C1^T."""
    say("nbf", nbf, "naux", naux, "na", na)
    B, packed, _, _ = inputs(nbf, naux, 1)
    rng = np.random.default_rng(4)
    C1, C2 = rng.standard_normal((2, na, nbf))

    def ints(B, C1, C2):
        R = np.einsum("bn,qmn,am->qba", C2, B, C1, optimize=True).reshape(naux, na * na)
        return R.T @ R

    with JKContext(nbf, naux, keep="fp64") as ctx:
        ctx.set_B_fitted(packed)
        for _ in range(2):
            got = ctx.active_ints(C1, C2).reshape(na * na, na * na)
            check(got, ints(B, C1, C2), ints(np.abs(B), np.abs(C1), np.abs(C2)), 4 * nbf + naux + 2)


@pytest.mark.parametrize("naux,nbf", [(1, 1), (16, 3), (63, 16), (64, 15), (65, 17), (130, 24), (200, 9)])
def test_fitted_tensor_at_block_edges(naux, nbf):
    """B = L^-1 (P|mn) from a metric of condition about ten: the error of a
    Cholesky factorisation and a substitution is below naux u cond(V) relative
    to the columns' norms (a factor 8 for the constants of both)."""
    say("naux", naux, "nbf", nbf)
    rng = np.random.default_rng(6)
    A = rng.standard_normal((naux, naux))
    V = A @ A.T / naux + np.eye(naux)
    T = rng.standard_normal((naux, nbf * (nbf + 1) // 2))
    want = np.linalg.solve(np.linalg.cholesky(V), T)
    with JKContext(nbf, naux, keep="fp64") as ctx:
        ctx.set_B(T, V)
        got = ctx.get_B()
    tol = 8.0 * naux * 2.0 ** -53 * np.linalg.cond(V) * np.linalg.norm(T, axis=0)
    say("  max error / bound", float(np.max(np.abs(got - want) / tol)))
    assert np.all(np.abs(got - want) <= tol)

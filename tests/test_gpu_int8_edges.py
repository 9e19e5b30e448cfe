"""The integer mode's kernels at the edges of their tiles, groups and dispatch
rules, against numpy in FP64: J and K of random B, D and C through the C-ABI,
each element held to the error bound of the digit arithmetic.

With r_Qm the largest |B_Qm:|, digits at the scale of a row leave out at most
2^-34 of its largest value (five digits, J) or 2^-27 (four, K; twice where the
packed triangle holds the value at the scale of the other row), and the digit
pairs that K's products drop sum to less than 1.01 2^-32 of the product of the
two rows' largest values per term. X is cut again at the scale of its largest
value over the orbitals and a pair of functions. FP64 sums add N u of the
absolute sums."""
import sys

import numpy as np
import pytest

from nopt_amd.jk import JKContext

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
# functions: 16-, 32- and 64-row tiles and slabs; auxiliary functions: pairs, the eighth per XCD; orbitals: 16-column
# tiles, one and two column groups. 176 and 192 functions: the last gamma partials that the J kernel adds itself, and
# the first that a kernel of their own does; 300 x 200: J and K on two streams.
SHAPES = [(1, 1, 1), (5, 2, 5), (16, 3, 16), (17, 15, 17), (31, 16, 2), (32, 17, 32), (33, 9, 33), (63, 7, 49),
          (65, 33, 65), (96, 5, 96), (97, 8, 97), (129, 6, 128), (161, 4, 160), (176, 40, 20), (192, 40, 20),
          (300, 200, 7)]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def inputs(nbf, naux, noccs, seed=5):
    rng = np.random.default_rng(seed)
    B = rng.standard_normal((naux, nbf, nbf)) * np.exp2(rng.integers(-3, 3, (naux, nbf, 1)))
    B = 0.5 * (B + B.transpose(0, 2, 1))
    B[:, nbf // 2:, : nbf // 4] = 0.0  # zero blocks
    B[:, : nbf // 4, nbf // 2:] = 0.0
    D = rng.standard_normal((len(noccs), nbf, nbf))
    r, c = np.tril_indices(nbf)
    return B, np.ascontiguousarray(B[:, r, c]), 0.5 * (D + D.transpose(0, 2, 1)), \
        [rng.standard_normal((n, nbf)) for n in noccs]


def bounds(B, D, C):
    """J, K and their error bounds."""
    naux, nbf = B.shape[:2]
    a, r = np.abs(B), np.abs(B).max(axis=2)
    rr = np.maximum(r[:, :, None], r[:, None, :])
    g, ga, gd = (np.einsum("qmn,mn->q", x, d) for x, d in ((B, D), (a, np.abs(D)), (rr, np.abs(D))))
    J = np.einsum("qmn,q->mn", B, g)
    dJ = 2.0 ** -34 * (1 + 2.0 ** -30) * (np.einsum("qmn,q->mn", rr, ga) + np.einsum("qmn,q->mn", a, gd)) \
        + 2 * (nbf * nbf + naux + 2) * U * np.einsum("qmn,q->mn", a, ga)
    ca = np.abs(C)
    cm = ca.max(axis=1)
    X = np.einsum("qmn,in->qmi", B, C, optimize=True)
    Xa = np.einsum("qmn,in->qmi", a, ca, optimize=True)
    dX = 2.0 ** -27 * (np.einsum("qmn,in->qmi", r[:, :, None] + r[:, None, :], ca, optimize=True)
                       + a.sum(axis=2)[:, :, None] * cm) * (1 + 2.0 ** -25) \
        + 1.01 * 2.0 ** -32 * nbf * r[:, :, None] * cm + 2 * nbf * U * Xa
    top = (np.abs(X) + dX).max(axis=2)  # largest of a row and of its neighbour in the pair of functions
    pair = np.concatenate([top, np.zeros((naux % 2, nbf))]).reshape(-1, 2, nbf).max(axis=1)
    top = np.repeat(pair, 2, axis=0)[:naux]
    dX += 2.0 ** -27 * top[:, :, None]
    K = np.einsum("qmi,qni->mn", X, X, optimize=True)
    ax = np.abs(X) + dX
    dK = np.einsum("qmi,qni->mn", dX, ax, optimize=True)
    dK = dK + dK.T + 1.01 * 2.0 ** -32 * X.shape[2] * np.einsum("qm,qn->mn", top, top) \
        + 2 * (naux * X.shape[2] + 2) * U * np.einsum("qmi,qni->mn", ax, ax, optimize=True)
    return J, K, dJ, dK


def check(what, got, want, tol):
    say("  ", what, "max error / bound", float(np.max(np.abs(got - want) / tol)))
    assert np.all(np.abs(got - want) <= tol), what
    assert np.array_equal(got, got.T), what


@pytest.mark.parametrize("compact", [False, True])
@pytest.mark.parametrize("nbf,naux,nocc", SHAPES)
def test_int8_build_at_tile_edges(nbf, naux, nocc, compact):
    say("nbf", nbf, "naux", naux, "nocc", nocc, "compact", compact)
    noccs = [nocc, max(1, nbf // 3)]
    B, packed, D, C = inputs(nbf, naux, noccs)
    want = [bounds(B, d, c) for d, c in zip(D, C)]
    with JKContext(nbf, naux, keep="int8", compact=compact) as ctx:
        ctx.set_B_fitted(packed)
        J, K = ctx.build(D[0], C[0], prec="int8")
        check("J", J, want[0][0], want[0][2])
        check("K", K, want[0][1], want[0][3])
        pair = ctx.build_batch([(d, c, len(c)) for d, c in zip(D, C)], prec="int8")
        for x, w in zip(pair, want):
            check("J of two", x[0], w[0], w[2])
            check("K of two", x[1], w[1], w[3])

"""The J pass inside the launch of the first exchange against the J pass as a
launch of its own: a build with its phases timed runs every phase by itself, an
ordinary build of this size shares the launch where a split's gamma values fit
(320 FP64, 512 integer ones of all densities; the long ranges of auxiliary
functions lie on either side). The same sums in the same order: bit for bit."""
import numpy as np
import pytest

from nopt_amd.jk import JKContext

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 17000, 1), (3, 2600, 2), (3, 5200, 2), (24, 116, 5), (65, 33, 64), (72, 348, 15),
          (145, 90, 30), (300, 200, 7)]


@pytest.mark.parametrize("prec", ["fp64", "int8"])
@pytest.mark.parametrize("nbf,naux,nocc", SHAPES)
def test_shared_launch_equals_separate_ones(nbf, naux, nocc, prec):
    print("nbf", nbf, "naux", naux, "nocc", nocc, prec, flush=True)
    rng = np.random.default_rng(7)
    D = rng.standard_normal((3, nbf, nbf))
    D = D + D.transpose(0, 2, 1)
    items = [(D[0], rng.standard_normal((nocc, nbf)), nocc), (D[1], rng.standard_normal((max(1, nbf // 3), nbf)),
                                                             max(1, nbf // 3)), (D[2], D[2][:1].copy(), 1)]
    with JKContext(nbf, naux, keep=prec) as ctx:
        ctx.set_B_fitted(rng.standard_normal((naux, nbf * (nbf + 1) // 2)))
        for n in (1, 2, 3):
            ctx.set_timing(True)
            want = ctx.build_batch(items[:n], prec=prec)
            ctx.set_timing(False)
            for _ in range(2):
                for got, w in zip(ctx.build_batch(items[:n], prec=prec), want):
                    assert np.array_equal(got[0], w[0]), "J"
                    assert np.array_equal(got[1], w[1]), "K"

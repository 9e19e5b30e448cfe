"""FP64 builds of two to four densities with different orbital counts at the
edges of the kernels' tiles, every J and K against numpy to the bound of
test_gpu_fp64.py. With up to two densities gamma comes out of the half-transform,
by pairs of functions and tiles of pair rows: one function, odd last functions,
many pairs to a tile and many tiles to a pair; with more it is a pass of its own."""
import numpy as np
import pytest

from nopt_amd.jk import JKContext
from test_gpu_fp64 import check, inputs, jk, say

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 5, 2), (7, 33, 3), (17, 9, 16), (24, 116, 5), (63, 7, 33), (64, 3, 64), (65, 8, 40),
          (80, 13, 80), (130, 5, 100), (200, 11, 70)]


@pytest.mark.parametrize("nbf,naux,nocc", SHAPES)
def test_fp64_batches_at_tile_edges(nbf, naux, nocc):
    say("nbf", nbf, "naux", naux, "nocc", nocc)
    B, packed, _, _ = inputs(nbf, naux, 1)
    rng = np.random.default_rng(8)
    D = rng.standard_normal((4, nbf, nbf))
    D = D + D.transpose(0, 2, 1)
    counts = [nocc, max(1, nocc // 2 + 1), 1, min(nbf, nocc + 3)]
    items = [(D[d], rng.standard_normal((n, nbf)), n) for d, n in enumerate(counts)]
    with JKContext(nbf, naux, keep="fp64") as ctx:
        ctx.set_B_fitted(packed)
        for nd in (2, 3, 4):
            for (J, K), (Dd, C, n) in zip(ctx.build_batch(items[:nd], prec="fp64"), items):
                J0, K0 = jk(B, Dd, C)
                Ja, Ka = jk(np.abs(B), np.abs(Dd), np.abs(C))
                check(J, J0, Ja, nbf * nbf + naux + 2)
                check(K, K0, Ka, 2 * nbf + naux * n + 2)

"""gram_tile and the kernels that use it (updates of a diagonal tile by low-rank
tiles, of a band tile by one dense and one low-rank or by two low-rank tiles) at
their edges: ranks 1, 16, 17, 64, 65 and, past the blocks of a grid, 200 and 210;
tiles of 130, 200 and 450 rows (a last row group that is not full); band 1 and 2.
Random tiles whose singular values all lie far above acc, so nothing is truncated
and the factor is numpy's Cholesky factor: 4 NB roundings of a matrix of condition
below 10, bound 1e-11 relative."""
import numpy as np
import pytest

import hicma_tlr as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [1, 2])
@pytest.mark.parametrize("NB,ra,rb,rc", [(130, 1, 17, 3), (130, 16, 40, 9), (200, 65, 64, 20), (450, 200, 210, 12)])
def test_products(ctx, NB, ra, rb, rc, band):
    rng = np.random.default_rng(NB + ra)
    NT, cap = 4, NB // 2
    g = H.TLRMatrix(ctx, NT * NB, NB, cap, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    g.generate(1e-1, 1, 1)           # allocates; the tiles are overwritten below
    if band > 1:
        g.regenerate(band)
    A = np.zeros((NT * NB, NT * NB))
    rank = {(3, 0): ra, (2, 0): rb, (3, 1): rc, (1, 0): 3, (2, 1): 2, (3, 2): 1}
    for m in range(NT):
        for n in range(m + 1):
            if m - n < band:
                T = 0.2 / NB * rng.standard_normal((NB, NB))
                if m == n:
                    T = T + T.T + 2.0 * np.eye(NB)
                g.set_tile(m, n, np.asfortranarray(T).ravel(order="F"), 0)
            else:
                r = rank[m, n]
                U, V = 0.2 / NB * rng.standard_normal((NB, r)), rng.standard_normal((NB, r))
                g.set_tile(m, n, np.concatenate([U.ravel(order="F"), V.ravel(order="F")]), r)
                T = U @ V.T
            b = slice(m * NB, (m + 1) * NB), slice(n * NB, (n + 1) * NB)
            A[b] = T
            A[b[::-1]] = T.T
    assert g.potrf(1e-8, 0, cap) == 0
    L, Ln = np.tril(g.uncompress()), np.linalg.cholesky(A)
    g.close()
    assert np.linalg.norm(L - Ln) <= 1e-11 * np.linalg.norm(Ln)

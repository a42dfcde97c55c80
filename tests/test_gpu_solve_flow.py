"""k_solve_flow at the edges of its variants: rows per thread (tiles of 40, 512,
513, 1025, 2050 rows: 1, 1, 2, 4, 8), groups of 1, 2 and 4 right-hand sides and
a last group that is not full, band 1 and 2, low-rank shares of no column, of
part of a round and of several, ragged last tiles.  The factor is random (unit
lower tiles set through hicma_set_tile), so its inverses are formed by the
solve; a factor of HiCMA_dpotrf_L brings its own and loses them with
hicma_set_tile.  Against scipy on the uncompressed factor; both sides sum the
same products in another order, and the diagonal tiles multiply by an inverse
(condition below 10): 1e-12 relative."""
import numpy as np
import pytest
from scipy.linalg import solve_triangular

import hicma_tlr as H

pytestmark = pytest.mark.gpu


def random_factor(ctx, N, NB, cap, band, rank, seed):
    rng = np.random.default_rng(seed)
    g = H.TLRMatrix(ctx, N, NB, cap, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    g.generate(1e-1, 1, 1)           # allocates; the tiles are overwritten below
    if band > 1:
        g.regenerate(band)
    L = np.zeros((N, N))
    for m in range(g.NT):
        rm = min(NB, N - m * NB)
        for n in range(m + 1):
            if m - n < band:
                T = np.zeros((NB, NB))
                T[:rm] = rng.standard_normal((rm, NB)) / NB
                if m == n:
                    T = np.tril(T, -1) + np.diag(1.0 + rng.random(NB))
                    T[rm:], T[:, rm:] = 0.0, 0.0
                    T[rm:, rm:] = np.eye(NB - rm)
                g.set_tile(m, n, np.asfortranarray(T).ravel(order="F"), 0)
            else:
                r = rank(m, n)
                U, V = np.zeros((NB, r)), rng.standard_normal((NB, r)) / NB
                U[:rm] = rng.standard_normal((rm, r))
                g.set_tile(m, n, np.concatenate([U.ravel(order="F"), V.ravel(order="F")]), r)
                T = U @ V.T
            cols = min(NB, N - n * NB)
            L[m * NB:m * NB + rm, n * NB:n * NB + cols] = T[:rm, :cols]
    return g, L


@pytest.mark.parametrize("N,NB,cap,band,nrhs", [(230, 40, 20, 1, 1), (230, 40, 20, 2, 3), (1500, 512, 200, 1, 2),
                                                (1900, 513, 200, 2, 5), (3000, 1025, 150, 1, 1),
                                                (3000, 1025, 150, 2, 9), (4000, 2050, 60, 1, 4), (4000, 2050, 60, 2, 1)])
def test_random_factor(ctx, N, NB, cap, band, nrhs):
    ranks = [0, 3, 17, cap]
    g, L = random_factor(ctx, N, NB, cap, band, lambda m, n: ranks[(m + 2 * n) % 4], seed=N + band)
    B = np.random.default_rng(nrhs).standard_normal((N, nrhs))
    for trans in (0, 1):
        want = solve_triangular(L, B, lower=True, trans=trans)
        got = g.trsm(B, trans)
        assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want), trans
        np.testing.assert_array_equal(g.trsm(B, trans), got)
    g.close()


def test_kept_inverses_follow_the_factor(ctx):
    N, NB, U = 1000, 200, 100
    g = H.TLRMatrix(ctx, N, NB, U, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    h = H.TLRMatrix(ctx, N, NB, U, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    b = np.random.default_rng(3).standard_normal(N)

    def check(A):
        L = np.tril(A.uncompress())
        want = solve_triangular(L, b, lower=True)
        got = A.trsm(b, 0)
        assert np.linalg.norm(got - want) <= 1e-11 * np.linalg.norm(want)
        return got

    assert g.generate(1e-8, U, 1) == 0 and g.potrf(1e-8, 0, U) == 0
    y = check(g)
    h.copy_from(g)                       # the copy brings the inverses
    np.testing.assert_array_equal(check(h), y)
    T, _ = g.get_tile(2, 2)
    h.set_tile(2, 2, np.asfortranarray(2.0 * T).ravel(order="F"), 0)  # and loses them
    assert np.linalg.norm(check(h) - y) > 1e-3 * np.linalg.norm(y)
    assert g.generate(1e-8, U, 1, params=(4.0, 0.1, 1e-2)) == 0 and g.potrf(1e-8, 0, U) == 0
    assert np.linalg.norm(check(g) - y) > 1e-3 * np.linalg.norm(y)
    g.close()
    h.close()

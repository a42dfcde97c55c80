"""k_rc_big at the edges of its variants: rows per thread of the QR panels
(tiles of 256, 257, 520, 1030 rows: 1, 2, 4 and 8), lanes per pair of the
Jacobi and whether its columns stay in LDS (stacks of 70 .. 570 columns), a
last panel of one column, r_B above the one-wave kernels' 64.  The three-tile
problem of test_gpu_rank_deficient (every singular value far above acc, so
only the capacity NB / 2 truncates, in the 290 + 280 case) against the same
steps in numpy, with that test's bound: 1e-9 relative, some 1e3 roundings
of the largest stack times cond(L) ~ 10."""
import numpy as np
import pytest

import hicma_tlr as H
from test_gpu_rank_deficient import build, load

pytestmark = pytest.mark.gpu
EPS = 1e-8


@pytest.mark.parametrize("NB,rc,ra,rb", [(256, 40, 30, 70), (256, 70, 58, 20), (257, 72, 57, 20), (300, 100, 61, 33),
                                         (520, 130, 131, 40), (600, 290, 280, 100), (1030, 60, 37, 20)])
def test_wide_stacks(ctx, NB, rc, ra, rb):
    tiles, A = build(NB, rc, ra, rb, seed=NB + rc)
    N, cap = 3 * NB, NB // 2
    g = H.TLRMatrix(ctx, N, NB, cap, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    g.generate(EPS, cap, 1)          # allocates the band; every tile is overwritten below
    load(g, tiles)
    assert g.potrf(EPS, 0, cap) == 0
    assert g.jacobi_unconverged() == 0
    L = np.tril(g.uncompress())
    Ln = np.zeros_like(A)
    b = [slice(i * NB, (i + 1) * NB) for i in range(3)]
    for i in range(3):
        Ln[b[i], b[i]] = np.linalg.cholesky(A[b[i], b[i]] - Ln[b[i], :i * NB] @ Ln[b[i], :i * NB].T)
        for m in range(i + 1, 3):
            C = A[b[m], b[i]] - Ln[b[m], :i * NB] @ Ln[b[i], :i * NB].T
            u, s, vt = np.linalg.svd(C)
            C = (u[:, :cap] * s[:cap]) @ vt[:cap]
            Ln[b[m], b[i]] = np.linalg.solve(Ln[b[i], b[i]], C.T).T
    (U, V), r = g.get_tile(2, 1)
    g.close()
    assert np.linalg.norm(L - Ln) <= 1e-9 * np.linalg.norm(Ln)
    # the trsm of step 1 multiplied V by L_11^-1, close to I / 2: U keeps
    # orthogonal columns, the singular values in descending order
    S = np.linalg.norm(U, axis=0)
    assert np.all(np.diff(S) <= 1e-12 * S[0])
    assert np.abs(U.T @ U - np.diag(S * S)).max() <= 1e-11 * S[0] ** 2

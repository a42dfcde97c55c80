"""k_compress_wg at the edges of its variants: rows per thread of the QR panels
(tiles of 250, 257, 520, 1030 rows), sketches of 64, 160 and the full width
(the ladder reaches the third pass on 3-D exp tiles, whose ranks pass 150),
ragged last tiles, and every covariance.  Each tile against the exact one:
||D - U V^T|| <= 3 tol ||D|| (the tail rule's tol, and the sketch's loss,
bounded by twice that as in the generation test of the CTest problem), and the
rank within 2 of the rank of the SVD by the same rule; a tile whose rank passes
the limits (half of its rows, maxrank) is refused with info -1."""
import numpy as np
import pytest

import hicma_tlr as H
import tlr_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,NB,U,kind,beta,tol", [(950, 250, 124, H.SQEXP_2D, 0.1, 1e-8),
                                                  (1000, 257, 128, H.SQEXP_2D, 0.1, 1e-6),
                                                  (1536, 512, 256, H.EXP_3D, 0.1, 1e-8),
                                                  (1500, 520, 255, H.SQEXP_3D, 0.05, 1e-5),
                                                  (3090, 1030, 300, H.SQEXP_2D, 0.05, 1e-8)])
def test_tiles(ctx, N, NB, U, kind, beta, tol):
    g = H.TLRMatrix(ctx, N, NB, U, kind, 1.0, beta, 1e-2, 3)
    info = g.generate(tol, U, 1)
    A = O.Oracle(N, NB, kind, 1.0, beta, 1e-2, 3).dense_exact()
    refused = 0
    for m in range(1, g.NT):
        for n in range(m):
            r = int(g.rank_map()[m, n])
            rows = min(NB, N - m * NB)
            D = A[m * NB:m * NB + rows, n * NB:(n + 1) * NB]
            s = np.linalg.svd(D, compute_uv=False)
            tail = np.sqrt(np.cumsum((s * s)[::-1])[::-1])
            want = int((tail > tol * tail[0]).sum())
            limit = min((min(rows, NB) + 1) // 2 - 1, U)   # largest rank that is stored: r < min / 2, r <= U
            if r == -1:
                refused += 1
                assert want + 2 > limit
                continue
            assert want - 2 <= limit
            (Um, Vm), r = g.get_tile(m, n)
            err = np.linalg.norm(Um[:rows] @ Vm.T - D)
            print(f"tile ({m},{n}) rank {r} (svd {want}) error {err / tail[0]:.2e}")
            assert abs(r - want) <= 2
            assert err <= 3 * tol * tail[0]
            assert np.all(Um[rows:] == 0.0) or np.abs(Um[rows:]).max() <= 1e-14
    assert info == (-1 if refused else 0)
    g.close()

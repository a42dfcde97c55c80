"""k_tile_normf over band tiles whose rows and columns are no multiple of a
wave's 32 columns or 256 rows, with a ragged last tile whose padding is left out,
against numpy: sums of up to 513^2 squares in another order, 1e-13 relative."""
import numpy as np
import pytest

import hicma_tlr as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,NB", [(76, 33), (520, 257), (1030, 513)])
def test_band_tiles(ctx, N, NB):
    rng = np.random.default_rng(N)
    g = H.TLRMatrix(ctx, N, NB, NB // 2, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    g.generate(1e-1, 1, 1)           # allocates; the tiles are overwritten below
    g.regenerate(2)
    want = {}
    for m in range(g.NT):
        for n in range(max(0, m - 1), m + 1):
            T = rng.standard_normal((NB, NB))
            if m == n:
                T = T + T.T
            g.set_tile(m, n, np.asfortranarray(T).ravel(order="F"), 0)
            want[m, n] = np.linalg.norm(T[:min(NB, N - m * NB), :min(NB, N - n * NB)])
    _, T = g.normf(tiles=True)
    g.close()
    for (m, n), w in want.items():
        assert abs(T[m, n] - w) <= 1e-13 * w, (m, n)

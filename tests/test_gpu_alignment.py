"""Tile sizes and rank capacities that put the diagonal tile's inverse blocks
(and the tiles' own columns) anywhere within a 128-byte line: the blocks that
k_potrf_dag passes between workgroups then share lines.  The factor against
numpy's dense Cholesky of the same matrix: the forward error is the
truncations (1e-8 each, a few tiles) amplified by cond(Sigma) ~ 1e4, so 1e-4
relative separates it from a stale block (errors of order 1)."""
import numpy as np
import pytest

import hicma_tlr as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,NB,U", [(768, 256, 127), (765, 255, 126), (825, 275, 136), (1395, 465, 231),
                                    (2700, 270, 135)])
def test_blocks_sharing_lines(ctx, N, NB, U):
    g = H.TLRMatrix(ctx, N, NB, U, H.SQEXP_2D, 1.0, 0.1, 1e-2, 0)
    assert g.generate(1e-8, U, 1) == 0
    D = np.tril(g.uncompress())
    want = np.linalg.cholesky(D + np.tril(D, -1).T)
    assert g.potrf(1e-8, 0, U) == 0
    got = np.tril(g.uncompress())
    g.close()
    assert np.linalg.norm(got - want) <= 1e-4 * np.linalg.norm(want)

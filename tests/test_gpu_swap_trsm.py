"""The interchanges and the triangular solve that follow a factored block, in
one pass (DLASWP and DTRSM of SRC/dgetrf.f:193-207), at the edges of its forms:
block widths around the 64-row solve blocks and the 16-row product tiles,
column counts around the 16 columns of a workgroup, a last block narrower than
the others, wide and tall matrices, leading dimensions past the matrix.

IPIV as the oracle's (near-ties traced), DGET01 < 30 (TESTING/dtest.in:13).
"""
import numpy as np
import pytest
import torch

import lapack_amd as la
import oracle

from gpu_util import ivec
from test_gpu_lu import THRESH, assert_ipiv, gpu_getrf

pytestmark = pytest.mark.gpu


@pytest.fixture
def tuning():
    yield la.set_tuning
    la.set_tuning(0, 0)


@pytest.mark.parametrize("nb,leaf", [(1, 1), (16, 16), (63, 64), (64, 64), (65, 64), (100, 64), (128, 32), (143, 64),
                                     (192, 64), (193, 48), (255, 64), (256, 64)])
def test_block_widths(dev, tuning, nb, leaf):
    tuning(nb, leaf)
    for m, n in [(nb + 1, nb + 1), (nb, nb + 17), (2 * nb + 15, 2 * nb + 1), (3 * nb + 5, nb + 33), (700, 3 * nb)]:
        a = la.matrix(2, 1000 * nb + m + n, m, n)
        lu_r, p_r, info_r = oracle.dgetrf(a)
        lu, p, info = gpu_getrf(a)
        assert info == info_r
        assert_ipiv(p, p_r, lu_r, lu)
        assert oracle.dget01(a, lu, p) < THRESH, (m, n)


def test_single_precision(dev, tuning):
    tuning(192, 64)
    for m, n in [(200, 457), (600, 600), (1300, 400)]:
        a = la.matrix(2, m + n, m, n).astype(np.float32)
        lu_r, p_r, info_r = oracle.sgetrf(a)
        lu, p, info = gpu_getrf(a, np.float32)
        assert info == info_r
        assert_ipiv(p, p_r, lu_r, lu, unit=2.0 ** -24)
        assert oracle.dget01(a.astype(np.float64), lu.astype(np.float64), p) * 2.0 ** -29 < THRESH


def test_leading_dimension_and_rows_past_the_matrix(dev):
    """lda > m: the rows past the matrix keep their bytes."""
    m, n, lda = 571, 390, 603
    a = la.matrix(2, 77, m, n)
    t = torch.full((n, lda), 7.25, dtype=torch.float64)
    t[:, :m] = torch.from_numpy(np.ascontiguousarray(a.T))
    d, p = t.cuda(), ivec(min(m, n))
    assert la.dgetrf(m, n, d, lda, p) == 0
    out = d.cpu().numpy()
    assert (out[:, m:] == 7.25).all()
    lu_r, p_r, _ = oracle.dgetrf(a)
    lu = np.asfortranarray(out[:, :m].T)
    assert_ipiv(p.cpu().numpy(), p_r, lu_r, lu)
    assert oracle.dget01(a, lu, p.cpu().numpy()) < THRESH

"""Host arrays through the synchronous entry points (SRC/dgesv.f:148): columns
that follow each other, and a leading dimension past the rows (packed through a
host buffer, several pieces for the largest): the same bits either way, and the
rows past the matrix keep theirs."""
import numpy as np
import pytest

import lapack_amd as la

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs,pad", [(1, 1, 3), (7, 5, 1), (130, 1, 70), (500, 4, 12), (2100, 3, 5)])
def test_strided_columns(dev, n, nrhs, pad):
    a, b = la.matrix(2, n, n, n), la.matrix(2, n + 1, n, nrhs)
    a0, b0, p0 = a.copy(order="F"), b.copy(order="F"), np.zeros(n, np.int32)
    assert la.dgesv(n, nrhs, a0, n, p0, b0, n) == 0
    lda, ldb = n + pad, n + 2 * pad
    a1, b1 = np.full((lda, n), 3.5, order="F"), np.full((ldb, nrhs), 4.5, order="F")
    a1[:n], b1[:n], p1 = a, b, np.zeros(n, np.int32)
    assert la.dgesv(n, nrhs, a1, lda, p1, b1, ldb) == 0
    np.testing.assert_array_equal(a1[:n], a0)
    np.testing.assert_array_equal(b1[:n], b0)
    np.testing.assert_array_equal(p1, p0)
    assert (a1[n:] == 3.5).all() and (b1[n:] == 4.5).all()

"""Host arrays through the synchronous entry points (SRC/dgesv.f:148): columns
that follow each other, and a leading dimension past the rows (packed through a
host buffer, several pieces for the largest): the same bits either way, and the
rows past the matrix keep theirs."""
import time

import numpy as np
import pytest
import torch

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


def host(n, ld, pinned):
    """An n-column array of ld rows, column-major, as a tensor of shape (n, ld)."""
    return torch.empty(n, ld, dtype=torch.float64, pin_memory=pinned)


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("m,n", [(3, 700), (24000, 40), (26000, 40), (1500, 300)])
def test_strided_routes(dev, pinned, m, n):
    """Columns shorter and longer than a packed copy is for, in pageable and in
    page-locked memory: the bits of contiguous columns, other rows untouched."""
    a = torch.from_numpy(la.matrix(2, m + n, m, n).T.copy())
    k = min(m, n)
    t0, p0 = a.clone(), np.zeros(k, np.int32)
    assert la.dgetrf(m, n, t0, m, p0) == 0
    t1, p1 = host(n, m + 9, pinned), np.zeros(k, np.int32)
    t1.fill_(2.5)
    t1[:, :m] = a
    assert la.dgetrf(m, n, t1, m + 9, p1) == 0
    assert torch.equal(t1[:, :m], t0) and bool((t1[:, m:] == 2.5).all())
    np.testing.assert_array_equal(p1, p0)


@pytest.mark.parametrize("m,n", [(20000, 200), (4000, 1000)])
def test_strided_page_locked_columns_go_as_fast_as_contiguous_ones(dev, m, n):
    """The bus moves page-locked columns at its full rate, strided or not; packed
    through a host buffer the call took more than twice as long."""
    best = {}
    for pad in (0, 8):
        t, p = host(n, m + pad, True), np.zeros(n, np.int32)
        src = torch.from_numpy(la.matrix(2, 5, m, n).T.copy())
        for _ in range(6):
            t[:, :m] = src
            t0 = time.perf_counter()
            assert la.dgetrf(m, n, t, m + pad, p) == 0
            best[pad] = min(best.get(pad, 1e9), time.perf_counter() - t0)
    assert best[8] < 1.4 * best[0], best

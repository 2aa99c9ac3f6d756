"""One right-hand side through DGETRS (SRC/dgetrs.f:181-218): the sweep by blocks of
128 rows, at the edges of its blocks, halves and 16-row parts, against the
oracle's DGETRS on the same factors and against the sweep that takes several
right-hand sides.

Tolerance: the matrices are random rows plus 4 sqrt(n) on the diagonal, their
rows shuffled, so that |L||U| stays a small multiple of |A| and the condition
number a small constant; every solution is then within a small multiple of
n eps of the exact one (Higham, Accuracy and Stability, thm 9.4), taken as
64 n eps.
"""
import numpy as np
import pytest
import torch

import lapack_amd as la
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 300, 385, 512, 513,
                               900])
def test_one_right_hand_side(dev, n, dtype):
    dbl = dtype == np.float64
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 4.0 * np.sqrt(n) * np.eye(n)
    a = np.asfortranarray(a[rng.permutation(n)].astype(dtype))
    lu, p = (oracle.dgetrf if dbl else oracle.sgetrf)(a)[:2]
    b = rng.standard_normal((n, 3)).astype(dtype)
    lda, ldb = n + 3, n + 5
    buf = np.full((n, lda), np.nan, dtype=dtype)  # what lies between n and lda is not read
    buf[:, :n] = lu.T
    d_a, d_p = torch.from_numpy(buf).cuda(), torch.from_numpy(np.asarray(p, dtype=np.int32)).cuda()
    tol = 64 * n * (2.0 ** -53 if dbl else 2.0 ** -24)
    for trans in "NT":
        ref = (oracle.dgetrs if dbl else oracle.sgetrs)(lu, p, np.asfortranarray(b), trans)[0]
        got = []
        for cols in ([0], [1], [0, 1, 2]):
            host = np.full((len(cols), ldb), 55.0, dtype=dtype)
            host[:, :n] = b[:, cols].T
            d_b = torch.from_numpy(host).cuda()
            rc = (la.dgetrs_async if dbl else la.sgetrs_async)(trans, n, len(cols), d_a, lda, d_p, d_b, ldb)
            torch.cuda.synchronize()
            assert rc == 0 and la.device_status() == 0
            out = d_b.cpu().numpy()
            assert (out[:, n:] == 55.0).all()
            got.append(out[:, :n])
        for x, r in ((got[0][0], ref[:, 0]), (got[1][0], ref[:, 1]), (got[0][0], got[2][0]), (got[1][0], got[2][1])):
            assert np.abs(x - r).max() <= tol * np.abs(r).max(), (n, trans)


@pytest.mark.parametrize("nrhs", [1, 3])
@pytest.mark.parametrize("n", [40, 100, 512, 513, 700])
def test_gesv_solves_only_the_nonsingular(dev, n, nrhs):
    """DGESV enqueues the solve behind the factorization: where INFO is not 0 it
    leaves B and the device's status alone (SRC/dgesv.f:170-175)."""
    rng = np.random.default_rng(n + nrhs)
    a = rng.standard_normal((n, n)) + 4.0 * np.sqrt(n) * np.eye(n)
    a = a[rng.permutation(n)]
    b = rng.standard_normal((n, nrhs))
    for singular in (False, True):
        m = a.copy()
        if singular:
            m[:, n // 2] = 0.0
        d_a, d_b = torch.from_numpy(m.T.copy()).cuda(), torch.from_numpy(b.T.copy()).cuda()
        d_p = torch.zeros(n, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        info = la.dgesv(n, nrhs, d_a, n, d_p, d_b, n)
        x = d_b.cpu().numpy().T
        assert la.device_status() == 0
        if singular:
            assert info == n // 2 + 1
            np.testing.assert_array_equal(x, b)
        else:
            assert info == 0
            assert oracle.dget02(np.asfortranarray(m), np.asfortranarray(x), np.asfortranarray(b)) < 30.0


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs", [1, 3, 16])
@pytest.mark.parametrize("n,zero", [(5, 2), (16, 15), (16, 0), (64, 40), (100, 55), (130, 66), (200, 199), (300, 150)])
def test_zero_on_the_diagonal(dev, n, zero, nrhs, dtype):
    """Factors with a zero on U's diagonal: what the substitution solves before it
    reaches the zero is not touched by it (BLAS/SRC/dtrsm.f:277-300), the row of the
    zero is not finite.  (Against A^T the second sweep takes it to every row.)"""
    dbl = dtype == np.float64
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 4.0 * np.sqrt(n) * np.eye(n)
    lu = (oracle.dgetrf if dbl else oracle.sgetrf)(np.asfortranarray(a.astype(dtype)))[0]
    lu[zero, zero] = 0
    p = np.arange(1, n + 1, dtype=np.int32)  # (rows stay in place)
    b = rng.standard_normal((n, nrhs)).astype(dtype)
    d_a, d_p = torch.from_numpy(np.ascontiguousarray(lu.T)).cuda(), torch.from_numpy(p).cuda()
    l, u = np.tril(lu.astype(np.float64), -1) + np.eye(n), np.triu(lu.astype(np.float64))
    tol = 64 * n * (2.0 ** -53 if dbl else 2.0 ** -24)
    d_b = torch.from_numpy(b.T.copy()).cuda()
    assert (la.dgetrs_async if dbl else la.sgetrs_async)("N", n, nrhs, d_a, n, d_p, d_b, n) == 0
    torch.cuda.synchronize()
    assert la.device_status() == 0
    x = d_b.cpu().numpy().T
    ref = np.linalg.solve(u[zero + 1:, zero + 1:], np.linalg.solve(l, b)[zero + 1:])
    assert not np.isfinite(x[zero]).any()
    if zero + 1 < n:
        assert np.abs(x[zero + 1:] - ref).max() <= tol * np.abs(ref).max()

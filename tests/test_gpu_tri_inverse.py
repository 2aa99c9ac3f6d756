"""The inverses of the 64 x 64 diagonal triangles in DGETRS's sweeps
(SRC/dgetrs.f:181-218): their error against 80 bits.

Right-hand sides that are unit vectors return the columns of the inverse.  The
yardstick is the inverse by doubling (2 x 2 block triangles of 1, 2, .., 32
rows, each product one chain of multiply-adds), in the same precision: over 60
triangles from LU factors of N(0,1) matrices the geometric mean of the error's
Frobenius norm may not exceed the yardstick's by more than 5 %.  (The standard
error of that mean is 2 to 3 %; emulated, the order of the sweeps' inverses gives 0.93 to
1.0.)
"""
import numpy as np
import pytest
import scipy.linalg as sl
import torch

import lapack_amd as la

pytestmark = pytest.mark.gpu

N = 64


def chain(a, b):
    """a b, every element one chain of fused multiply-adds (rounded through the next wider type)."""
    wide = np.longdouble if a.dtype == np.float64 else np.float64
    acc = np.zeros((a.shape[0], b.shape[1]), a.dtype)
    for k in range(a.shape[1]):
        acc = (np.outer(a[:, k].astype(wide), b[k].astype(wide)) + acc).astype(a.dtype)
    return acc


def by_doubling(m, lower, unit):
    v = m.copy()
    np.fill_diagonal(v, m.dtype.type(1) if unit else m.dtype.type(1) / np.diag(m))
    b = 1
    while b < N:
        for r in range(0, N, 2 * b):
            p, q = slice(r, r + b), slice(r + b, r + 2 * b)
            if lower:
                v[q, p] = -chain(v[q, q], chain(v[q, p], v[p, p]))
            else:
                v[p, q] = -chain(chain(v[p, p], v[p, q]), v[q, q])
        b *= 2
    return v


def exact(m, lower):
    m = m.astype(np.longdouble)
    v = np.eye(N, dtype=np.longdouble)
    for k in range(N) if lower else range(N - 1, -1, -1):
        v[k] /= m[k, k]
        below = slice(k + 1, N) if lower else slice(0, k)
        v[below] -= np.outer(m[below, k], v[k])
    return v


@pytest.mark.parametrize("nrhs", [1, 3, 16])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("factor,trans", [("U", "N"), ("U", "T"), ("L", "N"), ("L", "T")])
def test_error_of_the_inverse(dev, factor, trans, dtype, nrhs):
    dbl = dtype == np.float64
    d_p = torch.arange(1, N + 1, dtype=torch.int32, device="cuda")
    logs = []
    for seed in range(60):
        lu = sl.lu_factor(np.random.default_rng(seed).standard_normal((N, N)))[0]
        unit = factor == "L"
        m = (np.tril(lu, -1) + np.eye(N) if unit else np.triu(lu)).astype(dtype)  # (the other factor is I)
        d_a = torch.from_numpy(np.ascontiguousarray(m.T)).cuda()
        d_b = torch.eye(N, dtype=d_a.dtype, device="cuda")
        for c in range(0, N, nrhs):
            rc = (la.dgetrs_async if dbl else la.sgetrs_async)(trans, N, min(nrhs, N - c), d_a, N, d_p, d_b[c:], N)
            assert rc == 0
        torch.cuda.synchronize()
        t = np.ascontiguousarray(m.T) if trans == "T" else m
        lower = unit != (trans == "T")
        ref = exact(t, lower)

        def err(v):
            return float(np.sqrt(((v.astype(np.longdouble) - ref) ** 2).sum()))
        logs.append(np.log(err(d_b.cpu().numpy().T) / err(by_doubling(t, lower, unit))))
    assert np.exp(np.mean(logs)) <= 1.05

"""The batch's register form (orders up to 512) at the edges of its classes of
orders (64, 128, 256, 512 threads), of its blocks of 32 columns and of its
pieces of the columns to the right, against the oracle (SRC/dgetrf.f:105-225)
and against the panel form that a caller can select for the same matrices.

Bars: IPIV and INFO as the oracle's (near-ties traced), DGET01 < 30; what lies
between n and lda and past a matrix's pivots is not written.
"""
import numpy as np
import pytest
import torch

import lapack_amd as la
import oracle

from test_gpu_batched import THRESH, Batch, eps_of
from test_gpu_lu import assert_ipiv

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 95, 96, 97, 127, 128, 129, 160, 191, 255, 256,
         257, 289, 383, 447, 511, 512]


def factor(bt, plan):
    bt.d_a.copy_(bt.d_a0)
    bt.d_ipiv.fill_(-7)
    bt.d_info.fill_(-7)
    assert plan.getrf(bt.d_aptr, bt.d_lda, bt.d_pptr, bt.d_info) == 0
    torch.cuda.synchronize()
    return bt.d_a.cpu().numpy(), bt.d_ipiv.cpu().numpy(), bt.d_info.cpu().numpy()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["random", "zero_columns", "ties", "empty"])
def test_register_form(dev, kind, dtype):
    ns = ([0] + EDGES + [0]) if kind == "empty" else EDGES
    bt = Batch(ns, [1] * len(ns), 31, dtype, lda_pad=True)
    for k, (n, l, o) in enumerate(zip(ns, bt.ldas, bt.aoff)):
        a = bt.h_a[o:o + n * l].reshape(n, l)
        a[:, n:] = 77.0
        if kind == "zero_columns":
            for c in {0, n // 3, n - 1} if k % 3 == 0 else {min(n - 1, 33)} if k % 3 == 1 else set():
                a[c, :n] = 0.0
        elif kind == "ties":  # entries of +-1: equal candidates in the first columns
            a[:, :n] = np.sign(a[:, :n])
    bt.d_a0.copy_(torch.from_numpy(bt.h_a))
    plan = la.BatchPlan(ns, "d" if dtype == np.float64 else "s", autotune=False)
    assert plan.set_config(32, 512) == 0
    lu_all, piv_all, info_all = factor(bt, plan)
    assert plan.set_config(16, 256) == 0
    old_all, oldp_all, oldi_all = factor(bt, plan)
    np.testing.assert_array_equal(info_all, oldi_all)
    scale = 2.0 ** -53 / eps_of(dtype)  # the oracle's ratios are in units of 2^-53
    for k, (n, l, o) in enumerate(zip(ns, bt.ldas, bt.aoff)):
        if n == 0:
            assert info_all[k] == 0
            continue
        a = bt.a_host(k)
        lu = bt.a_host(k, lu_all)
        p, p_old = (v[k * bt.nmax:k * bt.nmax + bt.nmax] for v in (piv_all, oldp_all))
        assert (p[n:] == -7).all()
        assert (lu_all[o:o + n * l].reshape(n, l)[:, n:] == 77.0).all()
        if dtype == np.float64:
            lu_r, p_r, info_r = oracle.dgetrf(a)
        else:
            lu_r, p_r, info_r = oracle.sgetrf(a.astype(np.float32))
            lu_r = lu_r.astype(np.float64)
        if kind != "ties":  # later ties depend on the rounding of the products
            assert info_all[k] == info_r, (n, info_all[k], info_r)
            assert_ipiv(p[:n], p_r, lu_r, unit=eps_of(dtype))
        else:  # the first column has none: the first of the equal entries
            assert p[0] == p_r[0] == p_old[0] == 1
            assert (np.abs(np.tril(lu, -1)) <= 1.0).all()
        assert oracle.dget01(a, lu, p[:n]) * scale < THRESH, (kind, n)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["nan_below_the_head", "two_infinities"])
def test_zeros_right_of_a_block_that_is_not_finite(dev, kind, dtype):
    """DTRSM does not multiply a zero of the solution (BLAS/SRC/dtrsm.f:177-190):
    where L is not finite, a column right of the block whose rows of U are zero
    keeps them.  Infinities and NaNs lie where the panel form with blocks of the
    same 32 columns has them, IPIV and INFO are its."""
    ns = [33, 34, 48, 65, 100, 129, 200, 257, 300, 512]
    bt = Batch(ns, [1] * len(ns), 47, dtype)
    for k, (n, l, o) in enumerate(zip(ns, bt.ldas, bt.aoff)):
        a = bt.h_a[o:o + n * l].reshape(n, l)  # a[c, r] = A(r, c)
        if kind == "nan_below_the_head":
            a[3, n - 2] = np.nan
            a[7, 20] = np.nan
        else:  # the first becomes the pivot, the second's multiplier is inf / inf
            a[2, n // 2] = np.inf
            a[2, n - 1] = -np.inf
        for c in range(32, n, 3):  # columns of zeros, and of zeros in the first rows
            a[c, :n if c % 2 else min(n, 40)] = 0.0
    bt.d_a0.copy_(torch.from_numpy(bt.h_a))
    plan = la.BatchPlan(ns, "d" if dtype == np.float64 else "s", autotune=False)
    assert plan.set_config(32, 512) == 0
    lu_all, piv_all, info_all = factor(bt, plan)
    assert plan.set_config(32, 256) == 0
    old_all, oldp_all, oldi_all = factor(bt, plan)
    np.testing.assert_array_equal(info_all, oldi_all)
    for k, n in enumerate(ns):
        s = slice(k * bt.nmax, k * bt.nmax + n)
        np.testing.assert_array_equal(piv_all[s], oldp_all[s], err_msg=str(n))
        lu, old = bt.a_host(k, lu_all), bt.a_host(k, old_all)
        zero_rows = (old[:32, 32:] == 0).any()
        assert np.isnan(old[:, :32]).any() and zero_rows, n
        np.testing.assert_array_equal(np.isnan(lu), np.isnan(old), err_msg=str(n))
        np.testing.assert_array_equal(np.isinf(lu), np.isinf(old), err_msg=str(n))

"""The register-resident panel leaf (SRC/dgetrf2.f:179-214 column by column) at
the edges of its forms: the heights where the workgroup's size, the number of
workgroups and the single / multi-workgroup form change, and widths around the
8-column groups.

One column wide, a leaf is a pivot search, an interchange and a scaling, none
of which leaves room for rounding: IPIV, INFO and the column are bitwise the
oracle's, for ties, zeros, infinities, NaNs and subnormals as well.  Wider
leaves: IPIV as the oracle's (near-ties traced) and DGET01 < 30.
"""
import numpy as np
import pytest

import lapack_amd as la
import oracle

from test_gpu_lu import THRESH, assert_ipiv, gpu_getrf

pytestmark = pytest.mark.gpu

HEIGHTS = [1, 2, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 1537, 4097, 16385]


def column(kind, m, dtype, rng):
    a = rng.standard_normal(m)
    if kind == "ties":
        a = rng.integers(-2, 3, m).astype(float)
    elif kind == "zeros":
        a[:] = 0.0
    elif kind == "zero_but_last":
        a[:] = 0.0
        a[-1] = -3.0
    elif kind == "nan_head":
        a[0] = np.nan
    elif kind == "nan_inside":
        a[m // 2:] = np.nan
        a[0] = 0.5
    elif kind == "inf":
        a[m // 3] = np.inf
        a[-1] = -np.inf
    elif kind == "low_word":  # equal upper halves: the lower words decide
        a = 1.0 + rng.integers(0, 5, m) * np.finfo(dtype).eps
    elif kind == "tiny":
        a = a * float(np.finfo(dtype).tiny) / 8
    return np.asfortranarray(a.astype(dtype).reshape(m, 1))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["random", "ties", "zeros", "zero_but_last", "nan_head", "nan_inside", "inf",
                                  "low_word", "tiny"])
def test_one_column_bitwise(dev, kind, dtype):
    ref = oracle.dgetrf if dtype == np.float64 else oracle.sgetrf
    for m in HEIGHTS:
        a = column(kind, m, dtype, np.random.default_rng(m))
        lu_r, p_r, info_r = ref(a)
        lu, p, info = gpu_getrf(a, dtype)
        assert (info, p[0]) == (info_r, p_r[0]), (m, info, info_r, p, p_r)
        np.testing.assert_array_equal(lu, lu_r, err_msg=f"m = {m}")


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("w", [2, 7, 8, 9, 31, 33, 63, 64])
def test_leaf_against_oracle(dev, w, dtype):
    dbl = dtype == np.float64
    for m in HEIGHTS:
        if m < 2:
            continue
        a = la.matrix(2, 100 * m + w, m, w).astype(dtype)
        lu_r, p_r, info_r = (oracle.dgetrf if dbl else oracle.sgetrf)(a)
        lu, p, info = gpu_getrf(a, dtype)
        assert info == info_r
        assert_ipiv(p, p_r, lu_r, lu, unit=2.0 ** -53 if dbl else 2.0 ** -24)
        if dbl:
            assert oracle.dget01(a, lu, p) < THRESH
        else:
            # DGET01's ratio with the single precision's epsilon
            assert oracle.dget01(a.astype(np.float64), lu.astype(np.float64), p) * 2.0 ** -29 < THRESH


def test_zero_columns_inside_groups(dev):
    """Exact zero pivots at a group's first, inner and last columns: INFO is the
    first one, and the columns after it are factored like the oracle's."""
    for m in (100, 700, 2000):
        a = la.matrix(2, 9 + m, m, 40)
        for c in (8, 13, 23):
            a[:, c] = 0.0
        lu_r, p_r, info_r = oracle.dgetrf(a)
        lu, p, info = gpu_getrf(a)
        assert info == info_r == 9
        assert_ipiv(p, p_r, lu_r, lu)
        assert oracle.dget01(a, lu, p) < THRESH

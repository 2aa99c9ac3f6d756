"""The panel leaf's exchanges between workgroups at the heights where their form
changes: up to 8 workgroups (4096 rows) a wave polls one candidate a lane, up to
16 (8192 rows) two, and past that a workgroup folds its own first.  Cases and
bars are those of the leaf's own tests (test_gpu_leaf.py)."""
import numpy as np
import pytest

import lapack_amd as la
import oracle

from test_gpu_leaf import column
from test_gpu_lu import THRESH, assert_ipiv, gpu_getrf

pytestmark = pytest.mark.gpu

HEIGHTS = [513, 3585, 4096, 4097, 4608, 4609, 7681, 8192, 8193]


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
@pytest.mark.parametrize("w", [2, 9, 64])
def test_leaf_against_oracle(dev, w, dtype):
    dbl = dtype == np.float64
    for m in HEIGHTS:
        a = la.matrix(2, 100 * m + w, m, w).astype(dtype)
        a[:, w // 2] = np.where(np.arange(m) % 3 == 0, a[:, w // 2], 0)  # zeros among the candidates
        lu_r, p_r, info_r = (oracle.dgetrf if dbl else oracle.sgetrf)(a)
        lu, p, info = gpu_getrf(a, dtype)
        assert info == info_r
        assert_ipiv(p, p_r, lu_r, lu, unit=2.0 ** -53 if dbl else 2.0 ** -24)
        scale = 1.0 if dbl else 2.0 ** -29  # DGET01's ratio with the single precision's epsilon
        assert oracle.dget01(a.astype(np.float64), lu.astype(np.float64), p) * scale < THRESH

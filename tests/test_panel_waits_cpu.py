"""Which leaves of a factorization wait for another workgroup (CPU only).

A matrix of up to 1024 rows is factored by one workgroup a leaf: a
stream-ordered call of that size ends without a bounded wait, whatever else
runs on the GPU.  Taller matrices have leaves of several workgroups that agree
on each pivot.
"""
import ctypes

import pytest

import lapack_amd as la


@pytest.fixture(scope="module")
def groups():
    fn = getattr(ctypes.CDLL(la.LIB_PATH), "_ZN2la12panel_groupsEii")  # la::panel_groups(h, m); 0: one workgroup
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_int, ctypes.c_int]
    return fn


@pytest.mark.parametrize("m", [1, 512, 513, 600, 777, 1000, 1023, 1024])
def test_up_to_1024_rows_one_workgroup(groups, m):
    assert {groups(h, m) for h in range(1, m + 1)} == {0}


@pytest.mark.parametrize("m", [1025, 4096, 16384, 32768])
def test_taller_ones_a_workgroup_per_512_rows(groups, m):
    for h in {1, 512, 513, 1024, 1025, m}:
        assert groups(h, m) == (0 if h <= 512 else (h + 511) // 512)

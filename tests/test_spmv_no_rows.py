"""Dense SpMV of a matrix without rows: entries in it are malformed, and none is an empty sum."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import combblas_amd as cb


def _matrix(k, alloc):
    """0 x k with one entry per column, its arrays from alloc(values)."""
    keep = [alloc(np.arange(k + 1, dtype=np.int64)), alloc(np.arange(k, dtype=np.int64)),
            alloc(np.zeros(k, np.int64)), alloc(np.ones(k))]
    s = cb.cbx_dcsc(0, k, k, k, *[a[1] for a in keep], cb.DTYPES["float64"], cb.DEVICE)
    return s, keep


def _run(s, x):
    return cb.lib().cbx_spmv_dense(C.byref(s), x, None, cb.SEMIRINGS["plus_times"], cb.DTYPES["float64"], None)


@pytest.mark.parametrize("k", [1, 65535, 65536, 200_000])
def test_entries_without_rows_are_refused_before_the_device(k):
    def host(a):
        return a, a.ctypes.data

    s, keep = _matrix(k, host)
    x = np.ones(k)
    assert _run(s, x.ctypes.data) == cb.ERR_INVALID


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 65536])
def test_entries_without_rows_on_the_device(k):
    def device(a):
        d = cb.DeviceArray.from_host(a)
        return d, d.ptr

    s, keep = _matrix(k, device)
    x = cb.DeviceArray.from_host(np.ones(k))
    assert _run(s, x.ptr) == cb.ERR_INVALID
    none = cb.cbx_dcsc(0, k, 0, 0, keep[0][1], keep[1][1], keep[2][1], keep[3][1], cb.DTYPES["float64"], cb.DEVICE)
    assert _run(none, x.ptr) == cb.OK

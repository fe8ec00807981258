"""The mirror's slab layout, written and read back by k_ell_place / k_ell_scan.

Shapes at the edges: one row, 63 to 65 rows (a tile is 64), slot counts around the
tile's 16, the longest rows of one tile strip, every slab height, no slots, a
matrix wider than tall, and one of more entries than are staged at a time (64 MiB
at 12 bytes).  Copies are exact and the row products add slot by slot with separate
multiply and add, so both comparisons are for equality.
"""
import ctypes as C

import numpy as np
import pytest

from madmax_amd import _lib

pytestmark = pytest.mark.gpu


def matrix(n, ncol, nnz, seed):
    rng = np.random.default_rng(seed)
    cols = rng.integers(0, ncol, (n, nnz)).astype(np.int32)
    vals = rng.standard_normal((n, nnz))
    cut = rng.integers(0, nnz + 1, n)  # a row ends at its first -1; what follows is kept but not used
    cut[::3] = nnz
    cols[np.arange(n)[cut < nnz], cut[cut < nnz]] = -1
    return cols, vals


def create(cols, vals, ncol, slab):
    n, w = cols.shape
    m = _lib.EllMatrix(n, ncol, w, cols.ctypes.data_as(_lib.ip), vals.ctypes.data_as(_lib.dp))
    h = C.c_void_p()
    return m, h, _lib.lib().ell_device_create(C.byref(m), slab, C.byref(h))


def product(cols, vals, x):
    y = np.zeros(cols.shape[0])
    live = np.ones(cols.shape[0], bool)
    for j in range(cols.shape[1]):
        live &= cols[:, j] != -1
        y = np.where(live, y + vals[:, j] * x[np.maximum(cols[:, j], 0)], y)
    return y


@pytest.mark.parametrize("n,ncol,nnz,slab", [
    (1, 1, 1, 0), (63, 63, 15, 64), (64, 64, 16, 64), (65, 65, 17, 64), (257, 257, 0, 0), (300, 900, 33, 128),
    (1025, 1025, 81, 1024), (513, 40, 31, 256), (5, 7, 20000, 64), (70001, 70001, 81, 0),
])
def test_layout_round_trip(n, ncol, nnz, slab):
    lib = _lib.lib()
    cols, vals = matrix(n, ncol, nnz, n + nnz)
    print("ell layout: rows", n, "columns", ncol, "slots", nnz, "slab", slab, flush=True)
    m, h, rc = create(cols, vals, ncol, slab)
    assert rc == 0
    try:
        x = np.random.default_rng(0).standard_normal(ncol)
        for again in range(2):
            if again:  # the same shape, other entries
                cols2, vals2 = matrix(n, ncol, nnz, n + nnz + 1)
                cols[:], vals[:] = cols2, vals2
                assert lib.ell_device_update(h, C.byref(m)) == 0
            gc, gv, y = np.full_like(cols, -7), np.full_like(vals, np.nan), np.zeros(n)
            assert lib.ell_device_download(h, gc.ctypes.data_as(_lib.ip), gv.ctypes.data_as(_lib.dp)) == 0
            assert np.array_equal(gc, cols) and np.array_equal(gv, vals)
            assert lib.ell_device_mvp(h, x.ctypes.data_as(_lib.dp), y.ctypes.data_as(_lib.dp)) == 0
            assert np.array_equal(y, product(cols, vals, x))
    finally:
        lib.ell_device_destroy(h)


@pytest.mark.parametrize("bad", [-2, 50, 2**31 - 1, -2**31])
def test_refused_columns_leave_the_mirror(bad):
    lib = _lib.lib()
    cols, vals = matrix(50, 50, 9, 3)
    m, h, rc = create(cols, vals, 50, 0)
    assert rc == 0
    try:
        was = cols.copy()
        cols[49, 8] = bad
        assert create(cols, vals, 50, 0)[2] == 1
        assert lib.ell_device_update(h, C.byref(m)) == 1
        gc, gv = np.zeros_like(cols), np.zeros_like(vals)
        assert lib.ell_device_download(h, gc.ctypes.data_as(_lib.ip), gv.ctypes.data_as(_lib.dp)) == 0
        assert np.array_equal(gc, was)
    finally:
        lib.ell_device_destroy(h)

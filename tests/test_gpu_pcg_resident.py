"""The Jacobi-PCG with the matrix on chip (k_pcg_resident) against the two-launch
iteration and the CPU.

Shapes are where it could go wrong: one row, one row more than a slab, rows of
different lengths and an empty tail, the 81 slots it takes and one more, spans of
1,536 columns and the next that list theirs, columns spanning a slab's LDS for two
workgroups per CU, for one, and beyond it, the most slabs it takes and one more.  The fused kernel works on the same 256-row slabs in
the same order and rounds alike, so the bits are equal; x is also held against
numpy's residual: the solve stops at ||r|| <= 1e-10 ||b|| by the recurrence, and
the true residual of these well-conditioned systems (diagonally dominant by a
factor of two) follows it to the rounding of the row sums, 100 terms at 1e-16 of
|A||x| each: 1e-10 + 1e-13, checked at 2e-10.
"""
import ctypes as C
import threading

import numpy as np
import pytest

from madmax_amd import _lib

pytestmark = pytest.mark.gpu


def system(n, width, reach, seed):
    """Symmetric and diagonally dominant, `width` - 1 off-diagonal slots at most, columns up to `reach` away."""
    rng = np.random.default_rng(seed)
    half = max((width - 1) // 2, 0)
    offs = np.unique(np.concatenate([[min(reach, n - 1)], rng.integers(1, max(min(reach, n - 1), 1) + 1, half)]))
    offs = offs[(offs > 0) & (offs < n)][-half:] if half else np.zeros(0, int)
    cols = np.full((n, width), -1, np.int32)
    vals = np.zeros((n, width))
    fill = np.zeros(n, int)
    diag = np.ones(n)

    def put(r, c, v):
        cols[r, fill[r]] = c
        vals[r, fill[r]] = v
        fill[r] += 1

    up = [rng.uniform(-1, 0, n) * (rng.random(n) < 0.9) for _ in offs]
    for r in range(n):
        for o, w in zip(offs, up):
            if r - o >= 0 and w[r - o] != 0.0:
                put(r, r - o, w[r - o])
            if r + o < n and w[r] != 0.0:
                put(r, r + o, w[r])
        diag[r] += 2 * np.abs(vals[r]).sum()
        put(r, r, diag[r])
    return cols, vals, rng.standard_normal(n)


class Mirror:
    def __init__(self, cols, vals):
        self.cols, self.vals = np.ascontiguousarray(cols), np.ascontiguousarray(vals)
        n, w = cols.shape
        self.m = _lib.EllMatrix(n, n, w, self.cols.ctypes.data_as(_lib.ip), self.vals.ctypes.data_as(_lib.dp))
        self.h = C.c_void_p()
        assert _lib.lib().ell_device_create(C.byref(self.m), 0, C.byref(self.h)) == 0

    def solve(self, b, x0, fused):
        lib = _lib.lib()
        assert lib.ell_device_set_pcg_fused(self.h, fused) == 0
        x, s = x0.copy(), _lib.EllSolver(500, 0, 1e-10, 0.0)
        rc = lib.ell_device_solve_pcg(self.h, C.byref(s), b.ctypes.data_as(_lib.dp), x.ctypes.data_as(_lib.dp))
        return x, s.its, s.err, rc

    def close(self):
        _lib.lib().ell_device_destroy(self.h)


def residual(cols, vals, b, x):
    y = (np.where(cols >= 0, vals, 0.0) * x[np.maximum(cols, 0)]).sum(1)
    return np.linalg.norm(b - y) / np.linalg.norm(b)


@pytest.mark.parametrize("n,width,reach", [
    (1, 1, 1), (255, 5, 3), (257, 8, 200), (700, 81, 300), (700, 82, 300), (3993, 81, 500),
    (3000, 9, 640), (3000, 9, 642), (4000, 81, 1900),
    (12000, 27, 4700), (12000, 27, 9000), (20500, 9, 20400), (384 * 256, 9, 300), (384 * 256 + 1, 9, 300),
    (192 * 256 + 1, 9, 9000),
])
def test_matrix_on_chip_equals_other_mappings(n, width, reach):
    cols, vals, b = system(n, width, reach, 7 * n + width)
    print("resident pcg: rows", n, "slots", width, "reach", reach, flush=True)
    x0 = np.random.default_rng(1).standard_normal(n)
    m = Mirror(cols, vals)
    try:
        xa, ia, ea, ra = m.solve(b, x0, 0)
        xb, ib, eb, rb = m.solve(b, x0, 500)
    finally:
        m.close()
    assert ra == rb == 0 and ia == ib and ea == eb
    assert np.array_equal(xa, xb)
    assert residual(cols, vals, b, xa) < 2e-10


def test_concurrent_solves_share_the_chip():
    """Six threads, more workgroups together than run at once; each gets the bits it gets alone."""
    jobs = [system(n, 27, 4000, n) for n in (30000, 40000, 50000)] * 2
    mirrors = [Mirror(c, v) for c, v, _ in jobs]
    try:
        alone = [m.solve(j[2], np.zeros_like(j[2]), 0) for m, j in zip(mirrors, jobs)]
        got = [None] * len(jobs)

        def work(i):
            got[i] = mirrors[i].solve(jobs[i][2], np.zeros_like(jobs[i][2]), 0)

        ts = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    finally:
        for m in mirrors:
            m.close()
    for a, g in zip(alone, got):
        assert np.array_equal(a[0], g[0]) and a[1:] == g[1:] and a[3] == 0

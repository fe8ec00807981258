"""Whether a PCG solve has the matrix on chip: for the shapes that are to be solved
there, it is and does not fall back; past each limit it is not; and a mirror whose
workgroups cannot meet solves in two launches, tries again after a while and stays
when it can.  All mappings give the same bits, so the counts of the mirror say which
one ran.  (Compute units: the limits on the slabs follow from those of the device; the
shapes here are for 256.)"""
import ctypes as C
import threading

import numpy as np
import pytest

from madmax_amd import _lib
from tests.helpers import DevBuf
from tests.test_gpu_pcg_resident import Mirror, system

pytestmark = pytest.mark.gpu


def counts(m):
    out = (C.c_int * 3)()
    assert _lib.lib().ell_device_pcg_counts(m.h, out) == 0
    return tuple(out)


@pytest.mark.parametrize("n,width,reach,stays", [
    (1, 1, 1, True), (255, 5, 3, True), (257, 8, 200, True), (700, 81, 300, True), (700, 82, 300, False),
    (3993, 81, 500, True), (3000, 9, 640, True), (3000, 9, 642, True), (4000, 81, 1900, True),
    (12000, 27, 4700, True), (12000, 27, 9000, True), (20500, 9, 20400, False), (384 * 256, 9, 300, True),
    (384 * 256 + 1, 9, 300, False), (192 * 256, 9, 6000, True), (192 * 256 + 1, 9, 9000, False),
])
def test_which_solves_stay_on_chip(n, width, reach, stays):
    cols, vals, b = system(n, width, reach, 7 * n + width)
    print("rows", n, "slots", width, "reach", reach, flush=True)
    m = Mirror(cols, vals)
    try:
        assert m.solve(b, np.zeros(n), 0)[3] == 0
        assert counts(m) == ((1, 0, 0) if stays else (0, 0, 0))
    finally:
        m.close()


def test_concurrent_solves_do_not_fall_back():
    """118, 157 and 192 slabs at one to a CU: each fits, no two of the threads' together do."""
    jobs = [system(n, 27, 4000, n) for n in (30000, 40000, 49000)] * 2
    mirrors = [Mirror(c, v) for c, v, _ in jobs]
    try:
        def work(i):
            for _ in range(3):
                mirrors[i].solve(jobs[i][2], np.zeros_like(jobs[i][2]), 0)

        ts = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert [counts(m) for m in mirrors] == [(3, 0, 0)] * len(jobs)
    finally:
        for m in mirrors:
            m.close()


@pytest.mark.parametrize("n,width,reach", [(2000, 27, 300), (5000, 27, 2000)])
def test_without_a_meeting(n, width, reach):
    """Same bits from two launches, x and the guess untouched by the attempt; 1, 3, 7, .. solves between attempts."""
    cols, vals, b = system(n, width, reach, n)
    lib = _lib.lib()
    x0 = np.random.default_rng(2).standard_normal(n)
    m, seen = Mirror(cols, vals), []
    bd, xd = DevBuf(b), DevBuf(x0)
    try:
        ref = m.solve(b, x0, 0)
        assert counts(m) == (1, 0, 0)
        assert lib.ell_device_set_stay_away(m.h, 1) == 0
        for i in range(13):
            got = m.solve(b, x0, 0)
            assert np.array_equal(got[0], ref[0]) and got[1:] == ref[1:]
            seen.append(counts(m)[1])
        # attempts at the first solve, after 1, and after 3 and 7 more
        assert seen == [1, 1, 2, 2, 2, 2, 3, 3, 3, 3, 3, 3, 3]
        s = _lib.EllSolver(500, 0, 1e-10, 0.0)
        assert lib.ell_device_solve_pcg_noalloc(m.h, C.byref(s), bd.ptr, xd.ptr) == 0
        assert np.array_equal(xd.get(), ref[0]) and counts(m)[1:] == (3, 0)
        assert lib.ell_device_set_stay_away(m.h, 0) == 0
        assert np.array_equal(m.solve(b, x0, 0)[0], ref[0]) and counts(m) == (2, 3, 0)
        assert np.array_equal(m.solve(b, x0, 0)[0], ref[0]) and counts(m) == (3, 3, 0)
    finally:
        bd.free()
        xd.free()
        m.close()

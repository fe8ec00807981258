"""A mirror's download beside an engine at work: it waits for its own stream, not for the
engine's launches, which take some 40 ms each here.  Downloads of one mirror on several
threads do not disturb each other.

The bar of 10 ms lies between the two: without a wait for the engine a download takes
some 2 ms, the time until a running sweep leaves a CU.  Streams share the process's four
hardware queues in turn, and one that shares the engine's waits for it whatever it does:
of six mirrors, made one after the other, at least two do not."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from madmax_amd import MM_TANGENT_UNIT, Engine, _lib, configs, unit_loads
from tests.test_gpu_ell_layout import create, matrix

pytestmark = pytest.mark.gpu


def _download(h, shape):
    cols, vals = np.empty(shape, np.int32), np.empty(shape)
    assert _lib.lib().ell_device_download(h, cols.ctypes.data_as(_lib.ip), vals.ctypes.data_as(_lib.dp)) == 0
    return cols, vals


def test_download_beside_an_engine_at_work():
    cols, vals = matrix(3000, 3000, 81, 1)
    specs, stop, medians = [configs.c2_spec(1, i) for i in range(128)], threading.Event(), []
    with Engine(nrhs=6, hbm_budget=8 << 30, max_rves=136, rtol=1e-9) as eng:
        mirrors = [create(cols, vals, 3000, 0) for _ in range(6)]
        assert all(rc == 0 for _, _, rc in mirrors)

        def work():
            while not stop.is_set():
                for i, s in enumerate(specs):
                    eng.submit(i + 1, s, unit_loads(), MM_TANGENT_UNIT)
                eng.drain()
                eng.poll()

        th = threading.Thread(target=work)
        th.start()
        try:
            time.sleep(0.3)
            for _, h, _ in mirrors:
                times = []
                for _ in range(11):
                    t = time.perf_counter()
                    got = _download(h, cols.shape)
                    times.append(time.perf_counter() - t)
                    assert np.array_equal(got[0], cols) and np.array_equal(got[1], vals)
                    time.sleep(0.005)
                medians.append(np.median(times))
        finally:
            stop.set()
            th.join()
    for _, h, _ in mirrors:
        _lib.lib().ell_device_destroy(h)
    print("download, medians:", ", ".join("%.2f ms" % (1e3 * t) for t in medians))
    assert sorted(medians)[1] < 0.010


def test_downloads_on_several_threads():
    cols, vals = matrix(20000, 20000, 81, 2)
    m, h, rc = create(cols, vals, 20000, 0)
    assert rc == 0
    same = []

    def work():
        for _ in range(5):
            got = _download(h, cols.shape)
            same.append(np.array_equal(got[0], cols) and np.array_equal(got[1], vals))

    ts = [threading.Thread(target=work) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    _lib.lib().ell_device_destroy(h)
    assert same == [True] * 20

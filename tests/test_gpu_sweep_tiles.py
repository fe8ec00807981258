"""The resident sweep where the workgroups of a load case share the rows of the
z-planes as well as the planes, and where a cluster is large enough to have to
meet before its first exchange: against the step-by-step kernels and the oracle.

Sizes: two shares of the rows and one plane each, rows that do not divide, cells
longer than a strip of 62 positions and wide enough that a share is a few rows, few
planes over many rows and the reverse, up to a cluster of some 200 workgroups.
Engines of few RVEs (max_rves) take other splits than engines of many.

Bars.  Both solvers stop at a relative residual of 1e-10.  They differ in the
grouping of dot products and row sums, so that iteration counts are compared only
as a guard against slower convergence, to within a tenth; tangents and stresses
meet the repository's 1e-8 bar against each other and, where the oracle takes no
longer than seconds, against it.
"""
import threading

import numpy as np
import pytest

from madmax_amd import (MM_PREC_FP64, MM_PREC_MIXED, MM_TANGENT_NONE, MM_TANGENT_UNIT, Engine, rve_spec, unit_loads)
from tests.helpers import normwise_rel, oracle_rve

pytestmark = pytest.mark.gpu

TOL = 1e-8
EPS = np.array([1e-3, 2e-4, -1e-4, 0.0, 3e-4, 0.0])


def _kw(precision, **kw):
    return dict(precision=precision, inner_rtol=1e-10 if precision == MM_PREC_FP64 else 1e-5, max_inner_its=5000,
                **{"hbm_budget": 1 << 30, **kw})


def _solve(eng, specs, loads, mode):
    for i, s in enumerate(specs):
        assert eng.submit(i + 1, s, loads, mode) == 0
    eng.drain()
    res = {r["id"]: r for r in eng.poll()}
    return [res[i + 1] for i in range(len(specs))]


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
@pytest.mark.parametrize("n", [(33, 34, 2), (37, 35, 5), (70, 40, 4), (130, 9, 6), (5, 300, 3), (34, 38, 21)])
def test_shared_rows(n, precision):
    print("shared rows", n, "precision", precision, flush=True)
    spec = rve_spec(n, [(0.45, 0.55, 0.3)])
    with Engine(nrhs=6, **_kw(precision, max_rves=64)) as eng:
        r = _solve(eng, [spec], unit_loads(), MM_TANGENT_UNIT)[0]
    with Engine(nrhs=6, sync_every_step=True, **_kw(precision, max_rves=64)) as eng:
        s = _solve(eng, [spec], unit_loads(), MM_TANGENT_UNIT)[0]
    assert r["status"] == 0 and s["status"] == 0 and r["sweeps"] == s["sweeps"]
    assert abs(r["pcg_its"] - s["pcg_its"]) <= 2 * r["sweeps"] + s["pcg_its"] // 10
    assert normwise_rel(r["c_tangent"], s["c_tangent"]) <= TOL
    if np.prod(n) < 9000:
        c_ref, _ = oracle_rve(spec)[0].c_tangent_unit(1e-3, 1e-12)
        assert normwise_rel(r["c_tangent"], c_ref) <= TOL


@pytest.mark.parametrize("precision,n,max_rves", [
    (MM_PREC_MIXED, (24, 22, 20), 4), (MM_PREC_MIXED, (44, 41, 39), 200), (MM_PREC_MIXED, (60, 52, 50), 4),
    (MM_PREC_MIXED, (82, 80, 78), 2), (MM_PREC_FP64, (30, 28, 26), 2), (MM_PREC_FP64, (50, 47, 45), 200),
])
def test_one_load_case(precision, n, max_rves):
    """Splits for time and splits for throughput, up to a cluster of most of the GPU."""
    print("one load case", n, "precision", precision, "max_rves", max_rves, flush=True)
    spec = rve_spec(n, [(0.45, 0.55, 0.3)])
    out = []
    for sync in (False, True):
        with Engine(nrhs=1, sync_every_step=sync, **_kw(precision, max_rves=max_rves)) as eng:
            out.append(_solve(eng, [spec], [EPS], MM_TANGENT_NONE)[0])
    r, s = out
    assert r["status"] == 0 and s["status"] == 0 and r["sweeps"] == s["sweeps"]
    assert abs(r["pcg_its"] - s["pcg_its"]) <= 2 * r["sweeps"] + s["pcg_its"] // 10
    assert normwise_rel(r["stress"], s["stress"]) <= TOL


def test_large_clusters_in_turn_and_side_by_side():
    """Clusters that cannot run together: several in one launch, and two engines on
    two threads whose launches compete for the CUs.  Each result has the bits it has
    alone."""
    specs = [rve_spec((72, 70, 68), [(0.45, 0.5 + 0.02 * i, 0.3)]) for i in range(3)]
    alone = []
    for s in specs:
        with Engine(nrhs=1, **_kw(MM_PREC_MIXED, max_rves=3)) as eng:
            alone.append(_solve(eng, [s], [EPS], MM_TANGENT_NONE)[0])
    print("three in one launch", flush=True)
    for streams in (1, 2):
        with Engine(nrhs=1, solver_streams=streams, **_kw(MM_PREC_MIXED, max_rves=3)) as eng:
            for a, b in zip(alone, _solve(eng, specs, [EPS], MM_TANGENT_NONE)):
                assert b["status"] == 0 and np.array_equal(a["stress"], b["stress"]) and a["pcg_its"] == b["pcg_its"]
    print("two engines", flush=True)
    engines = [Engine(nrhs=1, **_kw(MM_PREC_MIXED, max_rves=3)) for _ in range(2)]
    got = [None, None]

    def work(i):
        got[i] = _solve(engines[i], specs, [EPS], MM_TANGENT_NONE)

    try:
        ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    finally:
        for e in engines:
            e.close()
    for g in got:
        for a, b in zip(alone, g):
            assert b["status"] == 0 and np.array_equal(a["stress"], b["stress"]) and a["pcg_its"] == b["pcg_its"]

"""The resident sweep (a whole PCG sweep of a load case in one launch, z in LDS,
p, q and d in registers, clusters of workgroups that split the z-planes)
against the oracle and against the step-by-step kernels (sync_every_step), at
the sizes where its tiling changes: one interior node, one and two strips of 62
positions, several ranks, the widest plane that fits and the first that does
not, and cells that are long in z.

Bars.  Both solvers stop at a relative residual of 1e-10, so each tangent meets
the repository's 1e-8 bar against the oracle.  The step-by-step kernels agree
with each other to 1e-12 (only the grouping of dot products differs).  The
resident sweep evaluates the same recurrences with a product that takes the
planes above and below together and so rounds differently; the iteration counts,
which depend on rounding, are compared to within a tenth as a guard against a
recurrence that converges slower, not as a bar on the results."""
import numpy as np
import pytest

from madmax_amd import (MM_ELL_DICT, MM_ELL_FULL, MM_PREC_FP64, MM_PREC_MIXED, MM_TANGENT_FD, MM_TANGENT_NONE,
                        MM_TANGENT_UNIT, Engine, fd_loads, rve_spec, unit_loads)
from tests.helpers import normwise_rel, oracle_rve

pytestmark = pytest.mark.gpu

TOL = 1e-8
GB = 1 << 30

# elements per side: what the size reaches
SIZES = [(2, 2, 2), (2, 3, 9), (1, 4, 5),  # one interior node; a thin column; no interior
         (32, 3, 4),   # 62 positions: one full strip
         (10, 9, 6),   # 80 positions: two strips
         (9, 8, 40),   # many planes over few columns
         (20, 17, 11), (31, 32, 6), (32, 32, 3),  # several strips per wave; the widest planes
         (34, 33, 3)]  # wider: the rows shared too


def _solve(eng, specs, loads=None, mode=MM_TANGENT_UNIT):
    for i, s in enumerate(specs):
        assert eng.submit(i + 1, s, loads if loads is not None else unit_loads(), mode) == 0
    eng.drain()
    res = {r["id"]: r for r in eng.poll()}
    return [res[i + 1] for i in range(len(specs))]


def _kw(precision):
    return dict(precision=precision, hbm_budget=GB, max_rves=32,
                inner_rtol=1e-10 if precision == MM_PREC_FP64 else 1e-5)


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
@pytest.mark.parametrize("n", SIZES)
def test_resident_sweep_vs_oracle_and_steps(n, precision):
    print("resident sweep", n, "precision", precision, flush=True)
    spec = rve_spec(n, [(0.45, 0.55, 0.3)])
    with Engine(nrhs=6, **_kw(precision)) as eng:
        r = _solve(eng, [spec])[0]
    with Engine(nrhs=6, sync_every_step=True, **_kw(precision)) as eng:
        s = _solve(eng, [spec])[0]
    ref, _ = oracle_rve(spec)
    c_ref, _ = ref.c_tangent_unit(1e-3, 1e-12)
    assert r["status"] == 0 and s["status"] == 0
    assert normwise_rel(r["c_tangent"], c_ref) <= TOL
    assert normwise_rel(s["c_tangent"], c_ref) <= TOL
    assert r["sweeps"] == s["sweeps"]
    assert abs(r["pcg_its"] - s["pcg_its"]) <= 2 * r["sweeps"] + s["pcg_its"] // 10


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
def test_step_kernels_agree(precision):
    """Kernel A slab by slab and as a z-plane march with two run lengths, on
    the step-by-step path, where small cells use them."""
    specs = [rve_spec(8, [(0.45, 0.5, 0.3)]), rve_spec((12, 9, 7), [(0.4, 0.6, 0.25)])]
    out = {}
    for planes in (0, 8, 2):
        with Engine(nrhs=6, march_planes=planes, sync_every_step=True, **_kw(precision)) as eng:
            out[planes] = _solve(eng, specs)
    for i, s in enumerate(specs):
        c_ref, _ = oracle_rve(s)[0].c_tangent_unit(1e-3, 1e-12)
        for planes in out:
            assert out[planes][i]["status"] == 0
            assert normwise_rel(out[planes][i]["c_tangent"], c_ref) <= TOL
        assert normwise_rel(out[8][i]["c_tangent"], out[0][i]["c_tangent"]) <= 1e-12
        assert normwise_rel(out[2][i]["c_tangent"], out[0][i]["c_tangent"]) <= 1e-12


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
def test_resident_and_other_rves_in_one_batch(precision):
    """Cells of several splits (planes, planes and rows, one workgroup) share the
    launches, in one and two stream groups, full and dictionary storage, each with the bits
    it has alone."""
    specs = [rve_spec((24, 23, 12), [(0.5, 0.45, 0.3)]), rve_spec((40, 36, 3), [(0.5, 0.5, 0.3)]),
             rve_spec(7, [(0.4, 0.5, 0.25)])]
    alone = []
    for s in specs:
        with Engine(nrhs=6, **_kw(precision)) as eng:
            alone.append(_solve(eng, [s])[0])
    for streams, storage in ((1, MM_ELL_DICT), (2, MM_ELL_DICT), (2, MM_ELL_FULL)):
        with Engine(nrhs=6, solver_streams=streams, ell_storage=storage, **_kw(precision)) as eng:
            for a, b in zip(alone, _solve(eng, specs)):
                assert b["status"] == 0
                assert np.array_equal(a["c_tangent"], b["c_tangent"])
                assert a["pcg_its"] == b["pcg_its"]


@pytest.mark.parametrize("nrhs", [1, 7])
def test_resident_sweep_load_counts(nrhs):
    """One load, and the seven of a finite-difference tangent, several ranks."""
    spec = rve_spec((21, 22, 19), [(0.5, 0.5, 0.3)])
    eps = np.array([1e-3, 2e-4, -1e-4, 0.0, 3e-4, 0.0])
    ref, _ = oracle_rve(spec)
    with Engine(nrhs=nrhs, **_kw(MM_PREC_MIXED)) as eng:
        if nrhs == 1:
            r = _solve(eng, [spec], [eps], MM_TANGENT_NONE)[0]
        else:
            r = _solve(eng, [spec], fd_loads(eps), MM_TANGENT_FD)[0]
    assert r["status"] == 0
    out = ref.homog(eps, rtol=1e-12)
    assert normwise_rel(r["stress"][0], out["stress_ave"]) <= TOL


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
def test_resident_sweep_iteration_cap(precision):
    """max_inner_its ends a sweep of every load case at the same count as the
    step-by-step path, and the results after it agree."""
    spec = rve_spec((12, 10, 17), [(0.5, 0.5, 0.3)])
    kw = dict(_kw(precision), max_inner_its=7, max_sweeps=2)
    with Engine(nrhs=6, **kw) as eng:
        r = _solve(eng, [spec])[0]
    with Engine(nrhs=6, sync_every_step=True, **kw) as eng:
        s = _solve(eng, [spec])[0]
    assert r["status"] == s["status"] != 0
    assert r["pcg_its"] == s["pcg_its"] == 14 and r["sweeps"] == s["sweeps"] == 2
    # fourteen iterations from the same start: rounding of the dot products only
    assert normwise_rel(r["c_tangent"], s["c_tangent"]) <= (1e-12 if precision == MM_PREC_FP64 else 1e-6)

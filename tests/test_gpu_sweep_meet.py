"""Clusters of workgroups that cannot meet: the RVE goes on by kernels A and B.

The host keeps some or all load cases from meeting (mm_engine_set_meet_off), which ends
the wait at once; the solve has to come back, with the results of the step-by-step
path.  Both stop at a relative residual of 1e-10, so stresses and tangents meet the
repository's 1e-8 bar against each other.  A sweep that was called off for every load
case counts neither in the result nor against max_sweeps: the rest is what the
step-by-step path does, in as many sweeps.  One that ran for some counts; the others
need as many after it, and the number of sweeps after rounding differently may differ
by one where the last but one ends at the edge of the tolerance."""
import ctypes as C

import numpy as np
import pytest

from madmax_amd import (MM_GUESS_AFFINE, MM_GUESS_ZERO, MM_PREC_FP64, MM_PREC_MIXED, MM_TANGENT_NONE,
                        MM_TANGENT_UNIT, Engine, _lib, rve_spec, unit_loads)
from tests.helpers import normwise_rel
from tests.test_sweep_splits import split_meet

pytestmark = pytest.mark.gpu

TOL = 1e-8
EPS = np.array([1e-3, 2e-4, -1e-4, 0.0, 3e-4, 0.0])
EPS2 = np.array([0.8e-3, 5e-4, 2e-4, -4e-4, 1e-4, 1e-4])


def _kw(precision, **kw):
    return dict(precision=precision, inner_rtol=1e-10 if precision == MM_PREC_FP64 else 1e-5, max_inner_its=5000,
                **{"hbm_budget": 2 << 30, "max_rves": 4, **kw})


def _meet_off(eng, mask):
    assert _lib.lib().mm_engine_set_meet_off(eng.h, C.c_uint(mask)) == 0


def _solve(eng, specs, loads, mode, **kw):
    for i, s in enumerate(specs):
        assert eng.submit(i + 1, s, loads, mode, **{k: v + i if k == "warm_key" else v for k, v in kw.items()}) == 0
    eng.drain()
    res = {r["id"]: r for r in eng.poll()}
    return [res[i + 1] for i in range(len(specs))]


@pytest.mark.parametrize("guess", [MM_GUESS_AFFINE, MM_GUESS_ZERO])
@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
@pytest.mark.parametrize("n,meet", [((36, 34, 33), 2), ((24, 24, 24), 1)])
def test_no_meeting_one_load_case(n, meet, precision, guess):
    """Alone, then, stepped from the start, beside a cell of one workgroup (swept on chip in the launches that step the
    other), and the first one again from its kept displacements, when its cluster is tried again."""
    fp64 = precision == MM_PREC_FP64
    assert split_meet(n, fp64, 1, 4, 128, 256)[4] == meet and split_meet((5, 5, 5), fp64, 1, 4, 128, 256)[0] == 1
    big, small = rve_spec(n, [(0.45, 0.55, 0.3)]), rve_spec((5, 5, 5), [(0.5, 0.5, 0.3)])
    ref = []
    with Engine(nrhs=1, sync_every_step=True, **_kw(precision, initial_guess=guess)) as eng:
        ref += _solve(eng, [big, small], [EPS], MM_TANGENT_NONE, warm_key=1)
        ref += _solve(eng, [big], [EPS2], MM_TANGENT_NONE, warm_key=1, warm_start=1)
    sweeps = ref[0]["sweeps"]
    print("no meeting", n, "precision", precision, "guess", guess, flush=True)
    with Engine(nrhs=1, **_kw(precision, initial_guess=guess, max_sweeps=sweeps)) as eng:
        _meet_off(eng, 1)
        out = _solve(eng, [big], [EPS], MM_TANGENT_NONE)
        out += _solve(eng, [big, small], [EPS], MM_TANGENT_NONE, warm_key=1)
        out += _solve(eng, [big], [EPS2], MM_TANGENT_NONE, warm_key=1, warm_start=1)
    for r, s in zip(out, [ref[0]] + ref):
        assert r["status"] == s["status"] == 0
        assert r["sweeps"] == s["sweeps"]
        assert normwise_rel(r["stress"], s["stress"]) <= TOL


@pytest.mark.parametrize("mask", [0b000101, 0b111110, 0b111111])
@pytest.mark.parametrize("n,meet", [((50, 47, 45), 2), ((24, 24, 24), 1)])
def test_some_load_cases_do_not_meet(n, meet, mask):
    """The displacements of the load cases that ran are kept, in one and in two stream groups."""
    assert split_meet(n, False, 6, 4, 128, 256)[4] == meet
    spec = rve_spec(n, [(0.45, 0.55, 0.3)])
    with Engine(nrhs=6, sync_every_step=True, **_kw(MM_PREC_MIXED)) as eng:
        s = _solve(eng, [spec], unit_loads(), MM_TANGENT_UNIT)[0]
    for streams in (1, 2):
        print("mask", bin(mask), "streams", streams, flush=True)
        with Engine(nrhs=6, solver_streams=streams, **_kw(MM_PREC_MIXED)) as eng:
            _meet_off(eng, mask)
            r = _solve(eng, [spec], unit_loads(), MM_TANGENT_UNIT)[0]
        assert r["status"] == s["status"] == 0 and abs(r["sweeps"] - s["sweeps"]) <= 1
        assert normwise_rel(r["c_tangent"], s["c_tangent"]) <= TOL

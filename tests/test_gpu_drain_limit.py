"""A drain gives every RVE the launches that its sweeps may take."""
import pytest

from madmax_amd import MM_PREC_MIXED, MM_TANGENT_UNIT, Engine, rve_spec, unit_loads
from tests.test_sweep_splits import split

pytestmark = pytest.mark.gpu


def test_many_short_sweeps_in_long_launches():
    """Sweeps of a single iteration (steepest descent) and many of them: whole sweeps come five to a launch whatever
    steps_per_launch says, so a limit counted in steps_per_launch would end the drain too early."""
    n = (24, 24, 24)
    assert split(n, False, 6, 4)[0] > 0
    with Engine(nrhs=6, precision=MM_PREC_MIXED, hbm_budget=1 << 30, max_rves=4, max_inner_its=1, max_sweeps=1000,
                steps_per_launch=4000) as eng:
        assert eng.submit(1, rve_spec(n, [(0.45, 0.55, 0.3)]), unit_loads(), MM_TANGENT_UNIT) == 0
        eng.drain()
        r = eng.poll()[0]
    # whether it converged or not, it ended by its own rules
    assert r["sweeps"] > 5 * 64 and (r["status"] == 0) == (r["sweeps"] < 1000)

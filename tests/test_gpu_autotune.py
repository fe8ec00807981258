"""The autotuner judges candidates by what the engine runs: whole solves where RVEs are
swept on chip (the slab shape), kernel A's own time where all are stepped."""
import pytest

from madmax_amd import Engine, autotune, rve_spec

pytestmark = pytest.mark.gpu

BEAM = (3, 4200, 3)  # too long for a resident sweep


def _spec(n):
    x, y, z = (0.1 * i for i in n)
    return rve_spec(n, [(0.45 * x, 0.4 * y, 0.3 * max(x, y))], lengths=(x, y, z))


@pytest.mark.parametrize("n,swept", [((12, 11, 10), True), (BEAM, False)])
def test_candidates_are_judged_by_the_kernel_that_runs(n, swept):
    out = autotune.tune([_spec(n)] * 2, budget=4 << 30, use_cache=False)
    assert all(t["swept"] == swept for t in out["trials"])
    shapes = [t for t in out["trials"] if t["inner_rtol"] == autotune.BASE_INNER and
              t["march_planes"] == autotune.BASE_PLANES]
    assert {t["slab_nodes"] for t in shapes} == set(autotune.SLAB_NODES)
    chosen = next(t for t in shapes if t["slab_nodes"] == out["slab_nodes"])
    what = "seconds" if swept else "step_ms"
    assert chosen[what] == min(t[what] for t in shapes)


def test_which_cells_are_swept():
    with Engine(nrhs=6, hbm_budget=1 << 30, max_rves=8) as eng:
        assert eng.swept(_spec((12, 11, 10))) and not eng.swept(_spec(BEAM)) and not eng.swept(_spec((1, 4, 5)))
    with Engine(nrhs=6, hbm_budget=1 << 30, max_rves=8, sync_every_step=True) as eng:
        assert not eng.swept(_spec((12, 11, 10)))

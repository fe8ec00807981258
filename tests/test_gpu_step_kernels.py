"""The step kernels A, S, B and R as engines launch them, in graphs, of several cells and
in two stream groups, on cells that no resident sweep takes: beams longer than 4,096
elements across y, which kernel A marches, and beams too long in x for a tile, which it
takes slab by slab.  (Their elements are cubes and every boundary node is held, so that
some tens of iterations solve them.)  And batches of such cells with cells that are swept on chip, where every kernel
has to leave the others' cells alone.

Bars.  All solves stop at a relative residual of 1e-10: 1e-8 to a sparse FP64 solve on
the CPU (the oracle's assembly takes hours for a beam; here its element stiffness is
assembled by scipy).  Storage,
streams, graphs, totals summed once per cell and the company in a batch change no bit;
the length of a march groups the partial sums differently, 1e-12."""
import functools

import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.linalg import cg

from madmax_amd import (MM_ELL_FULL, MM_PREC_FP64, MM_PREC_MIXED, MM_TANGENT_UNIT, Engine, rve_spec,
                        spec_fibers, unit_loads)
from oracle import pyoracle as po
from tests.helpers import normwise_rel
from tests.test_sweep_splits import split

pytestmark = pytest.mark.gpu

TOL = 1e-8
STEPPED = [(3, 4200, 3), (1000, 4, 4), (4, 4150, 7)]
SWEPT = [(20, 18, 17), (9, 8, 7), (40, 36, 3)]


def _spec(n):
    """Cubes of side 1 / 10, a fiber over a part of the length or of the section."""
    x, y, z = (0.1 * i for i in n)
    return rve_spec(n, [(0.45 * x, 0.4 * y, 0.3 * max(x, y))], lengths=(x, y, z))


def _kw(precision, **kw):
    return dict(nrhs=6, precision=precision, hbm_budget=4 << 30, max_rves=16,
                inner_rtol=1e-10 if precision == MM_PREC_FP64 else 1e-5, **kw)


def _solve(cells, precision, **kw):
    with Engine(**_kw(precision, **kw)) as eng:
        for i, n in enumerate(cells):
            assert eng.submit(i + 1, _spec(n), unit_loads(), MM_TANGENT_UNIT) == 0
        eng.drain()
        res = {r["id"]: r for r in eng.poll()}
    return [res[i + 1] for i in range(len(cells))]


@functools.lru_cache(None)
def _reference(n):
    """The tangent from boundary values E X, interior equilibrium by CG to 1e-13 and
    sigma_i . e_j = u_i K u_j / V (Hill's lemma, exact for the discrete solution)."""
    spec = _spec(n)
    m = po.mesh(3, *n, spec.lx, spec.ly, spec.lz)
    phase = po.phase_map(m, spec_fibers(spec))
    h = (spec.lx / n[0], spec.ly / n[1], spec.lz / n[2])
    nx, ny, nz = (i + 1 for i in n)
    e = np.arange(n[0] * n[1] * n[2])
    n0 = e % n[0] + (e // n[0]) % n[1] * nx + e // (n[0] * n[1]) * nx * ny
    node = np.stack([n0, n0 + 1, n0 + nx + 1, n0 + nx], 1)
    node = np.concatenate([node, node + nx * ny], 1)
    dof = (3 * node[:, :, None] + np.arange(3)).reshape(len(e), 24)
    ke = np.stack([po.ke(3, h, spec.young[k], spec.poisson[k]) for k in range(2)])
    K = sp.coo_matrix((ke[phase].ravel(), (np.repeat(dof, 24, 1).ravel(), np.tile(dof, (1, 24)).ravel())),
                      shape=(3 * nx * ny * nz,) * 2).tocsr()
    i = np.arange(nx * ny * nz)
    at = np.stack([i % nx, i // nx % ny, i // (nx * ny)], 1)
    inside = np.repeat(np.all((at > 0) & (at < np.array([nx, ny, nz]) - 1), 1), 3)
    X = at * np.array(h)
    A, B = K[inside][:, inside], K[inside][:, ~inside]
    M = sp.diags(1.0 / A.diagonal())
    us = []
    for v in np.eye(6):
        E = np.array([[v[0], v[3] / 2, v[5] / 2], [v[3] / 2, v[1], v[4] / 2], [v[5] / 2, v[4] / 2, v[2]]])
        u = (X @ E).ravel()
        u[inside], info = cg(A, -(B @ u[~inside]), x0=u[inside], rtol=1e-13, maxiter=5000, M=M)
        assert info == 0
        us.append(u)
    us = np.array(us)
    return us @ (K @ us.T) / (spec.lx * spec.ly * spec.lz)


def _same(a, b):
    assert a["status"] == 0 and b["status"] == 0
    assert np.array_equal(a["c_tangent"], b["c_tangent"])
    assert a["pcg_its"] == b["pcg_its"] and a["sweeps"] == b["sweeps"]


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
def test_stepped_batch(precision):
    fp64 = precision == MM_PREC_FP64
    assert all(split(n, fp64, 6, 16)[0] == 0 for n in STEPPED)
    ref = _solve(STEPPED, precision)
    for n, r in zip(STEPPED, ref):
        assert r["status"] == 0 and r["pcg_its"] > 5
        assert normwise_rel(r["c_tangent"], _reference(n)) <= TOL, n
    variants = [dict(solver_streams=1), dict(use_graph=False), dict(big_slabs=1), dict(big_slabs=400),
                dict(ell_storage=MM_ELL_FULL), dict(ell_storage=MM_ELL_FULL, big_slabs=1),
                dict(sync_every_step=True)]
    for kw in variants:
        print("step kernels: precision", precision, kw, flush=True)
        for a, b in zip(ref, _solve(STEPPED, precision, **kw)):
            _same(a, b)
    for kw in [dict(march_planes=0), dict(march_planes=2), dict(march_planes=0, ell_storage=MM_ELL_FULL, big_slabs=1),
               dict(march_planes=2, ell_storage=MM_ELL_FULL, big_slabs=1)]:
        print("step kernels: precision", precision, kw, flush=True)
        for a, b in zip(ref, _solve(STEPPED, precision, **kw)):
            assert b["status"] == 0 and normwise_rel(b["c_tangent"], a["c_tangent"]) <= 1e-12


@pytest.mark.parametrize("precision", [MM_PREC_MIXED, MM_PREC_FP64])
def test_stepped_and_swept_cells_in_one_batch(precision):
    fp64 = precision == MM_PREC_FP64
    cells = [SWEPT[0], STEPPED[0], SWEPT[1], STEPPED[1], SWEPT[2]]
    assert [split(n, fp64, 6, 16)[0] > 0 for n in cells] == [True, False, True, False, True]
    alone = [_solve([n], precision)[0] for n in cells]
    for n, r in zip(cells, alone):
        assert normwise_rel(r["c_tangent"], _reference(n)) <= TOL, n
    for order in (cells, cells[::-1]):
        for kw in [dict(), dict(solver_streams=1), dict(use_graph=False), dict(big_slabs=1),
                   dict(ell_storage=MM_ELL_FULL)]:
            print("mixed batch: precision", precision, kw, flush=True)
            out = _solve(order, precision, **kw)
            for a, b in zip(alone, out if order is cells else out[::-1]):
                _same(a, b)

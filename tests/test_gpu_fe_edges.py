"""The element-assembly kernels at the sizes where their mapping changes (four
elements and sixteen nodes per workgroup, eight elements per wavefront, slabs of
256 rows, both ends of every axis of the torus) against the oracle: element
stiffness and ELL sums, residuals and strains bit for bit, periodic solves
within the repository's 1e-8 bar."""
import ctypes as C

import numpy as np
import pytest

from madmax_amd import Macro, Micro, rve_spec
from madmax_amd import _lib
from oracle import pyoracle as po
from tests.helpers import normwise_rel, oracle_rve, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 2, 2), (2, 3, 9), (3, 5, 2), (16, 2, 2), (5, 4, 7)])
def test_reassembled_ell_and_residual_bitexact(n):
    print("element path", n, flush=True)
    spec = rve_spec(n, [(0.45, 0.55, 0.3)], lengths=(1.0, 0.8, 1.3))
    ref, _ = oracle_rve(spec)
    cols_ref, vals_ref = ref.assemble()
    x = np.random.default_rng(3).standard_normal(cols_ref.shape[0]) * 1e-4
    r_ref, n_ref = ref.residual(x)
    with Micro(spec, linear_materials=0, nl_min_norm=1e-12, nl_max_its=1) as m:
        m.fe2(np.array([1e-3, 0, 2e-4, 0, 1e-4, 0]))
        cols, vals = m.ell()
        r, nrm = m.residual(x)
    assert np.array_equal(cols, cols_ref)
    assert same_bits(vals, vals_ref)
    assert same_bits(r, r_ref)
    assert abs(nrm - n_ref) <= 1e-13 * n_ref


@pytest.mark.parametrize("n", [(3, 3, 3), (3, 4, 5), (6, 3, 4)])
def test_periodic_solve_on_uneven_tori(n):
    spec = rve_spec(n, [(0.5, 0.45, 0.3)])
    ref, _ = oracle_rve(spec)
    eps = np.array([1e-3, 2e-4, -3e-4, 4e-4, -1e-4, 2e-4])
    print("torus", n, flush=True)
    with Micro(spec, rtol=1e-12, fe2_bc=_lib.MICRO_BC_PER_LM) as m:
        se, ss = m.fe2(eps)
        cols, _ = m.ell()
    out = ref.homog_per_lm(eps)
    assert normwise_rel(ss, out["stress_ave"]) <= 1e-8
    assert normwise_rel(se, eps) <= 1e-12
    # first-touch order: elements ascending, then their corners
    nx, ny, nz = n
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    order = [[] for _ in range(nx * ny * nz)]
    for e in range(nx * ny * nz):
        ex, ey, ez = e % nx, (e // nx) % ny, e // (nx * ny)
        nodes = [((ex + a) % nx) + ((ey + b) % ny) * nx + ((ez + c) % nz) * nx * ny for a, b, c in corner]
        for u in nodes:
            order[u] += [v for v in nodes if v not in order[u]]
    ref_cols = np.array([[3 * v + d for v in order[u] for d in range(3)] for u in range(len(order))])
    assert np.array_equal(cols[0::3], ref_cols)
    assert np.array_equal(cols[2::3], ref_cols)


@pytest.mark.parametrize("n", [1, 3])
def test_macro_tangents_with_zeros_and_full(n):
    """Tangents with zero entries (skipped for a whole wavefront) beside full
    ones: the element stiffness of each equals the oracle's bit for bit."""
    rng = np.random.default_rng(7)
    full = rng.standard_normal((6, 6)) * 1e6 + np.eye(6) * 1e8
    iso = po.material_c(3, 2e7, 0.28)
    c_gp = np.array([[iso if (e + g) % 3 else full for g in range(8)] for e in range(n ** 3)])
    with Macro(n) as m:
        m.set_dirichlet(np.zeros(0, dtype=np.int32))
        m.assemble_a(c_gp)
        cols, vals = m.ell()
        nrow = m.nrow
    nx = n + 1
    X = np.array([[ix, iy, iz] for iz in range(nx) for iy in range(nx) for ix in range(nx)], dtype=float) * (1.0 / n)
    K = po.OrEll()
    po.lib().or_ell_init(C.byref(K), nrow, nrow, 81)
    for e in range(n ** 3):
        n0 = e % n + ((e // n) % n) * nx + (e // (n * n)) * nx * nx
        nods = [n0, n0 + 1, n0 + nx + 1, n0 + nx]
        nods += [v + nx * nx for v in nods]
        idx = np.array([3 * a + d for a in nods for d in range(3)], dtype=np.int32)
        ke = po.macro_ke(X[nods], c_gp[e])
        po.lib().or_ell_add_vals(C.byref(K), po._p(idx, po.ip), 24, po._p(idx, po.ip), 24, po._p(ke))
    cols_ref, vals_ref = po.ell_to_numpy(K)
    po.lib().or_ell_free(C.byref(K))
    assert np.array_equal(cols, cols_ref)
    assert same_bits(vals, vals_ref)

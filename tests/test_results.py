"""Results of the C struct as dicts, one at a time and all at once: the same fields, types and values, in arrays that
do not share the struct's memory."""
import numpy as np

from madmax_amd import _lib
from madmax_amd.engine import Result, result_dict, result_dicts


def _filled(i):
    r = Result()
    r.id, r.status, r.pcg_its, r.sweeps, r.residual_rel = 7 + i, 5, 100 + i, 2, 1e-11 * (i + 1)
    r.t_submit, r.t_admit, r.t_done = 1.0, 2.0, 3.0 + i
    for k in range(_lib.MM_MAX_RHS):
        for j in range(6):
            r.stress[k][j], r.strain[k][j] = 100 * i + 10 * k + j, -(100 * i + 10 * k + j)
    for j in range(36):
        r.c_tangent[j] = 1000 * i + j
    return r


def test_one_and_many_results():
    buf = (Result * 5)(*[_filled(i) for i in range(5)])
    many = result_dicts(buf, 4, lambda rid: rid - 6)
    assert [m["id"] for m in many] == [7, 8, 9, 10] and result_dicts(buf, 0, None) == []
    for i, m in enumerate(many):
        r = _filled(i)
        one = result_dict(r, i + 1)
        for d in (m, one):
            assert type(d["id"]) is int and type(d["residual_rel"]) is float
            assert (d["status"], d["pcg_its"], d["sweeps"], d["residual_rel"]) == (5, 100 + i, 2, 1e-11 * (i + 1))
            assert (d["t_submit"], d["t_admit"], d["t_done"]) == (1.0, 2.0, 3.0 + i)
            for name, sign in (("stress", 1), ("strain", -1)):
                want = np.array([[sign * (100 * i + 10 * k + j) for j in range(6)] for k in range(i + 1)], float)
                assert d[name].dtype == np.float64 and np.array_equal(d[name], want) and d[name].flags.owndata
            assert np.array_equal(d["c_tangent"], (1000.0 * i + np.arange(36)).reshape(6, 6))
        r.stress[0][0] = -1
        assert one["stress"][0, 0] == 100 * i
    buf[0].c_tangent[0] = -1
    assert many[0]["c_tangent"][0, 0] == 0

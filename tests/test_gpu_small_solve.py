"""The one-workgroup solve of small natural-order systems against the same
solve by level-scheduled launches: the same bits, iterations and verdict, for
both sides of the rule's line, grids whose levels are one row, one chunk of 16
rows and more, every precision, exhausted iterations and a zero right-hand
side."""
import numpy as np
import pytest

import omodels_amd as om

pytestmark = pytest.mark.gpu

DAY = 86400.0
# 1536 rows: the largest of the rule where tiles exist; 1540: the next path
GRIDS = [(1, 1, 1), (2, 1, 1), (37, 1, 1), (16, 16, 1), (17, 3, 5), (10, 8, 6), (16, 12, 8), (20, 11, 7)]


def _solve(c, schedule, precision, zero=False, **kw):
    m = om.Model(c)
    m.set_solution(c.pv0, c.mean0)
    J, r = m.linearize(DAY, iteration_index=0)
    rng = np.random.default_rng(7)
    r = np.zeros_like(r) if zero else r + 1e-3 * np.abs(r).max() * rng.standard_normal(r.shape)
    s = om.Solver(m, om.default_params(ilu_schedule=schedule, precision=precision, **kw))
    s.prepare(J, r)
    rc, x, its = s.solve()
    return rc, np.array(x), its


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("grid", GRIDS)
def test_same_bits_as_launches(grid, precision):
    c = om.BlackOilCase(om.make_spec(*grid, seed=5))
    got, want = _solve(c, 0, precision), _solve(c, 1, precision)
    assert got[0] == want[0] and got[2] == want[2]
    assert np.array_equal(got[1], want[1])


@pytest.mark.parametrize("kw", [dict(lin_max_iter=1), dict(lin_max_iter=3), dict(lin_tol=1e-30, lin_abs_tol=0.0),
                                dict(zero=True), dict(lin_max_error=1e-30)])
def test_same_verdict_as_launches(kw):
    c = om.BlackOilCase(om.make_spec(9, 7, 4, seed=6))
    got, want = _solve(c, 0, 0, **kw), _solve(c, 1, 0, **kw)
    assert got[0] == want[0] and got[2] == want[2]
    assert np.array_equal(got[1], want[1])

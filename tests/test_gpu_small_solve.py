"""The one-workgroup factorization and solve of small natural-order systems
against the same by level-scheduled launches: the same bits, iterations and
verdict, for grids whose levels are one row, one chunk of 16 rows and more,
every precision, exhausted iterations and a zero right-hand side; on both sides
of the line where tiles exist (1536 rows), and up to the line elsewhere (FP32
systems and auxiliary rows: 16384 scalar rows, the workgroup's LDS) with the
next larger system, whose default is the launches themselves.  The 2x2 blocks
are held to the launches in test_gpu_lens.py."""
import numpy as np
import pytest

import omodels_amd as om
from cases import RateWell

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


# 5461 rows: the largest of the rule without tiles; 5462 and 5472: above it
@pytest.mark.parametrize("grid", [(43, 127, 1), (17, 17, 18), (16, 18, 19)])
def test_same_bits_at_the_largest_fp32_systems(grid):
    c = om.BlackOilCase(om.make_spec(*grid, seed=8))
    got, want = (_solve(c, sched, 2, lin_max_iter=30) for sched in (0, 1))
    assert got[0] == want[0] and got[2] == want[2]
    assert np.array_equal(got[1], want[1])


def _aux_solve(grid, schedule, precision, everywhere=False):
    """two wells as auxiliary rows; everywhere: the first linked to every cell
    of the grid, a row of many more blocks than the grid's"""
    c = om.BlackOilCase(om.make_spec(*grid, seed=9))
    nxy = grid[0] * grid[1]
    inj = list(range(c.N)) if everywhere else [I for I in range(c.N) if I % nxy == grid[0] + 1]
    prod = [I for I in range(c.N) if I % nxy == nxy - grid[0] - 2]
    rng = np.random.default_rng(9)
    well = RateWell(c.N, [(inj, rng.uniform(0.5e-9, 2e-9, len(inj)) / len(inj), 4.0),
                          (prod, rng.uniform(0.5e-9, 2e-9, len(prod)), -1.0)])
    m = om.Model(c)
    m.set_auxiliary(well.n_aux, *well.links())
    m.set_solution(c.pv0, c.mean0)
    aux = well.initial(c.pv0)
    m.set_auxiliary_solution(aux)
    m.linearize(DAY, iteration_index=0)
    m.add_auxiliary(*well.terms(c.pv0, c.mean0, aux))
    s = om.Solver(m, om.default_params(ilu_schedule=schedule, precision=precision, lin_max_iter=30))
    s.prepare()
    lu = s.ilu() if precision < 2 else None
    rc, x, its = s.solve()
    return rc, x, its, lu


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("grid,everywhere", [((5, 4, 3), True), ((12, 9, 6), True), ((16, 16, 16), False),
                                             ((53, 103, 1), False), ((42, 130, 1), False)])
def test_same_bits_with_auxiliary_rows(grid, everywhere, precision):
    got, want = (_aux_solve(grid, sched, precision, everywhere) for sched in (0, 1))
    assert got[0] == want[0] and got[2] == want[2]
    assert np.array_equal(got[1], want[1])
    if precision < 2:
        assert np.array_equal(got[3], want[3])

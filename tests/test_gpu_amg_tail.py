"""The V-cycle's small levels in one workgroup, and the coarse correction taken
by the first backward colour as it reads: one cycle against the oracle bit for
bit on grids whose levels lie on either side of the one-workgroup line (1024
cells), that are nothing but such levels, and without post-smoothing (the
correction is then a pass of its own)."""
import numpy as np
import pytest

import omodels_amd as om
import oracle as orc
from test_gpu_amg import _bits, _both, _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(16, 16, 4), (41, 5, 5), (11, 3, 1), (4, 4, 2), (31, 31, 30), (2, 520, 1)])
@pytest.mark.parametrize("kw", [dict(), dict(amg_pre_smooth=1, amg_post_smooth=0),
                                dict(amg_agg=(2, 2, 2), amg_coarsen_target=1, amg_post_smooth=1)])
def test_cycle_bit_exact_around_the_line(dims, kw):
    c, pat, J, r = _system(dims)
    prm, prmo = _both(**kw)
    s = om.Solver(om.Model(c), prm)
    s.prepare(J, r)
    d = np.random.default_rng(8).standard_normal(3 * c.N)
    rc, vo = orc.amg_apply(dims, pat["row_ptr"], pat["col_idx"], J, prmo, d)
    assert rc == 0
    for rep in range(2):
        assert np.array_equal(_bits(s.apply_precond(d)), _bits(vo)), rep

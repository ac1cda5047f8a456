"""The FP32 V-cycle bit for bit.  It runs only inside the FP32 inner solve, so
one BiCGStab iteration of that solve (two applications) is restated in numpy:
FP32 level matrices, vectors and element-wise steps, FP64 pivots and coarsest
inverse, exact scalar products rounded once.  In FP64 the restated cycle is
held to the oracle's, which is what makes it a reference.  The grids have all
their levels in one workgroup (at most 1024 cells), levels on either side of
that line, and one cell next to it; with and without post-smoothing."""
import math

import numpy as np
import pytest

import omodels_amd as om
import oracle as orc
from cases import case, mixed_state

GRIDS = [(11, 3, 1), (16, 16, 4), (41, 5, 5), (13, 19, 22)]
KW = [dict(), dict(amg_pre_smooth=1, amg_post_smooth=0),
      dict(amg_agg=(2, 2, 2), amg_coarsen_target=8, amg_pre_smooth=1, amg_post_smooth=1)]


def _system(dims, seed=3):
    c = case(*dims, seed=seed)
    prob = orc.problem_from_case(c)
    pv, mean = mixed_state(c, seed=seed)
    J, r = orc.linearize(prob, pv, mean, orc.storage(prob, *mixed_state(c, seed=seed + 1)), 43200.0)
    return c, orc.pattern(prob), J, r


def _block_inverse(a):
    """adjugate over determinant of [N][3][3], in the factorization's order of operations"""
    a = a.reshape(-1, 9).T
    c00, c01, c02 = a[4] * a[8] - a[5] * a[7], a[5] * a[6] - a[3] * a[8], a[3] * a[7] - a[4] * a[6]
    r = 1.0 / (a[0] * c00 + a[1] * c01 + a[2] * c02)
    c10, c11, c12 = a[2] * a[7] - a[1] * a[8], a[0] * a[8] - a[2] * a[6], a[1] * a[6] - a[0] * a[7]
    c20, c21, c22 = a[1] * a[5] - a[2] * a[4], a[2] * a[3] - a[0] * a[5], a[0] * a[4] - a[1] * a[3]
    return np.stack([c00 * r, c10 * r, c20 * r, c01 * r, c11 * r, c21 * r, c02 * r, c12 * r, c22 * r], 1).reshape(-1, 3, 3)


class _Level:
    def __init__(self, dims, A, dtype):
        nx, ny, nz = (int(v) for v in dims)
        self.dims, self.N = (nx, ny, nz), nx * ny * nz
        A = A.reshape(7, self.N, 3, 3)
        self.D, self.A, self.dinv = A[3], A.astype(dtype), _block_inverse(A[3])
        I = np.arange(self.N)
        self.ijk = i, j, k = I % nx, (I // nx) % ny, I // (nx * ny)
        self.even = (i + j + k) % 2 == 0
        self.nb = [(k > 0, -nx * ny), (j > 0, -nx), (i > 0, -1), (i >= 0, 0), (i + 1 < nx, 1), (j + 1 < ny, nx),
                   (k + 1 < nz, nx * ny)]

    def product(self, s, rows, x):
        """block of slot s times x, on the rows that have the neighbour"""
        rows = rows[self.nb[s][0][rows]]
        a, v = self.A[s, rows], x[rows + self.nb[s][1]]
        return rows, (a[:, :, 0] * v[:, None, 0] + a[:, :, 1] * v[:, None, 1]) + a[:, :, 2] * v[:, None, 2]

    def apply(self, x):
        y = np.zeros_like(x)
        for s in range(7):
            rows, p = self.product(s, np.arange(self.N), x)
            y[rows] += p
        return y

    def colour(self, b, x, even, skip=False):
        rows = np.nonzero(self.even == even)[0]
        acc = b.copy()
        for s in (0, 1, 2, 4, 5, 6):
            if not skip:
                r, p = self.product(s, rows, x)
                acc[r] -= p
        a, D = acc[rows].astype(np.float64), self.dinv[rows]
        o = (D[:, :, 0] * a[:, None, 0] + D[:, :, 1] * a[:, None, 1]) + D[:, :, 2] * a[:, None, 2]
        x[rows] = (0.0 + o).astype(x.dtype)

    def residual(self, b, x):
        rows = np.nonzero(self.even)[0]
        r = np.zeros_like(b)
        r[rows] = b[rows]
        for s in range(7):
            q, p = self.product(s, rows, x)
            r[q] -= p
        return r


class _Cycle:
    def __init__(self, dims, mats, kw, dtype):
        self.lv = [_Level(d, A, dtype) for d, A in zip(dims, mats)]
        self.agg = kw.get("amg_agg", (3, 3, 3))
        self.pre, self.post, self.damp = kw.get("amg_pre_smooth", 2), kw.get("amg_post_smooth", 2), dtype(1.6)
        C = self.lv[-1]
        M = np.zeros((C.N, 3, C.N, 3))
        A = mats[-1].reshape(7, C.N, 3, 3)
        for s in range(7):
            rows = np.nonzero(C.nb[s][0])[0]
            M[rows, :, rows + C.nb[s][1], :] = A[s, rows]
        rc, self.inv = orc.dense_inverse(M.reshape(3 * C.N, 3 * C.N))
        assert rc == 0

    def __call__(self, b, l=0):
        L = self.lv[l]
        if l + 1 == len(self.lv):
            d = b.ravel().astype(np.float64)
            s = self.inv[:, 0] * d[0]
            for j in range(1, d.size):
                s = s + self.inv[:, j] * d[j]
            return s.astype(b.dtype).reshape(-1, 3)
        x = np.zeros_like(b)
        for k in range(self.pre):
            L.colour(b, x, True, skip=k == 0)
            L.colour(b, x, False)
        r, C = L.residual(b, x), self.lv[l + 1]
        ai, aj, ak = (L.ijk[q] // self.agg[q] for q in range(3))
        of = ai + C.dims[0] * (aj + C.dims[1] * ak)
        bc = np.zeros((C.N, 3), b.dtype)
        for I in np.nonzero(L.even)[0]:          # a coarse cell's even cells in natural order
            bc[of[I]] += r[I]
        x += self.damp * self(bc, l + 1)[of]
        for k in range(self.post):
            L.colour(b, x, False)
            L.colour(b, x, True)
        return x


@pytest.mark.parametrize("kw", KW)
@pytest.mark.parametrize("dims", GRIDS)
def test_restated_cycle_is_the_oracles_in_fp64(dims, kw):
    c, pat, J, _ = _system(dims)
    prm = orc.amg_params(**kw)
    levels = orc.amg_dims(dims, prm)
    mats = [orc.amg_level_matrix(dims, pat["row_ptr"], pat["col_idx"], J, prm, l)[1] for l in range(len(levels))]
    d = np.random.default_rng(8).standard_normal(3 * c.N)
    rc, want = orc.amg_apply(dims, pat["row_ptr"], pat["col_idx"], J, prm, d)
    assert rc == 0
    got = _Cycle(levels, mats, kw, np.float64)(d.reshape(-1, 3)).ravel()
    assert np.array_equal(got.view(np.uint64), np.asarray(want).view(np.uint64))


@pytest.mark.gpu
@pytest.mark.parametrize("kw", KW)
@pytest.mark.parametrize("dims", GRIDS)
def test_one_fp32_iteration_is_the_restatements(dims, kw):
    c, pat, J, r0 = _system(dims)
    s = om.Solver(om.Model(c), om.default_params(precond=2, precision=1, lin_max_iter=1, lin_tol=1e-12, lin_abs_tol=0.0,
                                                 **kw))
    s.prepare(J, r0)
    rc, x, its = s.solve()
    assert rc == 1 and its == 1
    levels = s.amg_dims()
    M = _Cycle(levels, [s.amg_level(l) for l in range(len(levels))], kw, np.float32)
    A = M.lv[0].apply
    f32 = np.float32

    def dot(a, b):
        return math.fsum((a.astype(np.float64) * b.astype(np.float64)).ravel().tolist())

    b = r0.astype(f32).reshape(-1, 3)
    rho = dot(b, b)                     # p = r = b in the first iteration
    y = M(b)
    v = A(y)
    alpha = rho / dot(b, v)
    want = y * f32(alpha)
    r = b - v * f32(alpha)
    z = M(r)
    t = A(z)
    omega = dot(t, r) / dot(t, t)
    want = want + f32(omega) * z
    assert np.array_equal(x.view(np.uint64), want.ravel().astype(np.float64).view(np.uint64))

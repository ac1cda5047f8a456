"""The work that a user of this library has it do, as measured cases.

Four kinds of call, all through the Python binding of the C ABI:

  steps      Model.simulate: implicit time steps of one reservoir from its
             initial state (Newton loop, assembly, preconditioned BiCGStab)
  iteration  one Newton iteration by its pieces, as a simulator that keeps its
             own Newton loop calls the plugins (linearize, prepare, solve,
             update); "host": with the Jacobian and the residual handed over
             as host arrays, "report": followed by FLOWS / FLORES and the
             output quantities
  serve      requests of uneven size submitted to the continuous-batching
             server and served together
  lens       the two-phase immiscible lens problem to a given time

Options: order 0 (natural-order ILU(0)) or 1 (two-colour ILU(0)), precond 0
(ILU(0)) or 2 (aggregation AMG), precision 0 (FP64) or 1 (FP32 inner solve in
FP64 refinement), terms (diffusion, dispersion, rock compressibility).

Sizes are the ones of this repository's configurations, tests and benchmark
(40x40x10, 100x100x50, 120x120x30, 200x200x50, the 8k-250k cell requests) and
odd ones between them.
"""
import math
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.getcwd(), "opm-models_amd"))
import omodels_amd as om  # noqa: E402

DAY = 86400.0


def listed():
    return [
        # the smallest grid (the smoke run's): a coarse model or a sector, where
        # launches and latency are all there is
        dict(name="steps_480", kind="steps", nx=12, ny=10, nz=4, steps=3, order=0, precond=0, precision=0),
        # a 16k-cell reservoir at the reference's own settings
        dict(name="steps_16k", kind="steps", nx=40, ny=40, nz=10, steps=2, order=0, precond=0, precision=0),
        # the headline run: 500k cells, FP64, the reference's preconditioner
        dict(name="steps_500k", kind="steps", nx=100, ny=100, nz=50, steps=1, order=0, precond=0, precision=0),
        # the same grid in the mixed-precision form
        dict(name="steps_500k_fp32_two_colour", kind="steps", nx=100, ny=100, nz=50, steps=1, order=1, precond=0,
             precision=1),
        # the 432k-cell grid with the AMG in FP64 (half a day: for some fields a
        # whole day's step fails and is halved)
        dict(name="steps_432k_amg", kind="steps", nx=120, ny=120, nz=30, steps=1, dt_days=0.5, order=0, precond=2,
             precision=0),
        # the largest grid, 2M cells, with the AMG in the mixed-precision form
        # (its wells' rates grow with the pore volume: shorter steps)
        dict(name="steps_2m_fp32_amg", kind="steps", nx=200, ny=200, nz=50, steps=1, dt_days=0.1, order=0, precond=2,
             precision=1),
        # odd sizes with every optional term of the assembly
        dict(name="steps_54k_terms", kind="steps", nx=61, ny=47, nz=19, steps=1, order=0, precond=0, precision=0,
             terms=True),
        # the drop-in boundary: a simulator that passes host arrays both ways
        dict(name="iteration_98k_host", kind="iteration", nx=70, ny=70, nz=20, order=0, precond=0, precision=0,
             host=True, report=False),
        # device-resident pieces with a report's output, odd sizes, two colours
        dict(name="iteration_132k_report", kind="iteration", nx=83, ny=53, nz=30, order=1, precond=0, precision=0,
             host=False, report=True),
        # an ensemble request stream in the serving form
        dict(name="serve_8", kind="serve", requests=8, cells_min=8000, cells_max=60000, steps=2, order=1, precision=1),
        # an ensemble on the plain FP64 path
        dict(name="serve_6_natural", kind="serve", requests=6, cells_min=8000, cells_max=30000, steps=1, order=0,
             precision=0),
        # two-phase lens problem, the smallest systems (2x2 blocks)
        dict(name="lens_48x32", kind="lens", nx=48, ny=32, t_end=1000.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "iteration", "iteration", "serve", "lens"])
    if kind == "lens":
        return dict(kind="lens", nx=rng.randint(12, 64), ny=rng.randint(10, 40), t_end=float(rng.randint(5, 10) * 100))
    if kind == "serve":
        lo = int(_log(rng, 2000, 10000))
        return dict(kind="serve", requests=rng.randint(2, 8), cells_min=lo, cells_max=lo * rng.randint(2, 5),
                    steps=1, order=rng.choice([0, 1]), precision=rng.choice([0, 1]))
    n = _log(rng, 400, 300000)
    nz = max(2, min(60, int(round(_log(rng, 3, 40) * (n / 30000.0) ** 0.2))))
    nx = max(3, int(round(math.sqrt(n / nz) * rng.uniform(0.5, 2.0))))
    ny = max(3, int(round(n / nz / nx)))
    order, precond = rng.choice([(0, 0), (0, 0), (1, 0), (0, 2)])
    precision = rng.choice([0, 0, 1])
    if kind == "steps":
        return dict(kind="steps", nx=nx, ny=ny, nz=nz, steps=1, order=order, precond=precond, precision=precision,
                    terms=rng.random() < 0.3)
    return dict(kind="iteration", nx=nx, ny=ny, nz=nz, order=order, precond=precond, precision=precision,
                host=rng.random() < 0.3, report=rng.random() < 0.3)


# ---------------------------------------------------------------------------
def _params(case):
    """Steps of at most a day (the benchmark's and the requests') unless the
    case says otherwise; everything else the reference's values."""
    return om.default_params(max_dt=DAY * case.get("dt_days", 1.0), ilu_order=case["order"], precond=case.get("precond", 0),
                             precision=case["precision"])


def _reservoir(case, seed):
    return om.BlackOilCase(om.make_spec(case["nx"], case["ny"], case["nz"], seed=seed))


def _disturbed(c, seed):
    """A state in the middle of a run: water and pressure moved, free gas in
    some cells and undersaturated oil in others."""
    rng = np.random.default_rng(seed)
    pv, mean = c.pv0.copy(), c.mean0.copy()
    pv[1::3] *= 1.0 + 0.002 * rng.standard_normal(c.N)
    pv[0::3] += 0.1 * rng.random(c.N)
    gas = rng.random(c.N) < 0.2
    mean[gas] = 0
    pv[2::3][gas] = 0.05 * rng.random(int(gas.sum()))
    pv[2::3][~gas] *= 0.95 + 0.04 * rng.random(int((~gas).sum()))
    return pv, mean


def _request_cases(case, seed):
    rng = np.random.default_rng(seed)
    sizes = np.random.default_rng(case["requests"])
    out = []
    for k in range(case["requests"]):
        n = sizes.uniform(case["cells_min"], case["cells_max"])
        nz = int(sizes.integers(5, 16))
        nxy = max(4, int(round(math.sqrt(n / nz))))
        out.append(om.BlackOilCase(om.make_spec(nxy, nxy, nz, seed=seed * 101 + k, wells=2,
                                                perm_sigma=float(rng.uniform(0.5, 1.5)))))
    return out


def _lens_problem(case, seed):
    rng = np.random.default_rng(seed)
    return om.lens_problem(nx=case["nx"], ny=case["ny"], k_lens=1e-12 * float(rng.uniform(0.8, 1.25)),
                           k_outer=1e-10 * float(rng.uniform(0.8, 1.25)), porosity=float(rng.uniform(0.36, 0.44)))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "steps":
        c = _reservoir(case, seed)
        m = om.Model(c)
        if case.get("terms"):
            rng = np.random.default_rng(seed + 1)
            m.set_diffusion(1e-9, 2e-9, mw_oil=0.2, mw_gas=0.02)
            m.set_dispersion(cell_dispersion=0.01 * rng.random(c.N))
            m.set_rock(comp=1e-10 * (0.5 + rng.random(c.N)), pref=np.full(c.N, 200e5))
        return dict(case=case, res=c, model=m, params=_params(case))
    if kind == "iteration":
        c = _reservoir(case, seed)
        m = om.Model(c)
        prm = _params(case)
        pv, mean = _disturbed(c, seed + 1)
        return dict(case=case, res=c, model=m, params=prm, solver=om.Solver(m, prm), pv=pv, mean=mean)
    if kind == "serve":
        return dict(case=case, requests=_request_cases(case, seed), server=om.Server(_params(case), 64 * 2.0 ** 30, 64))
    p = _lens_problem(case, seed)
    m = om.LensModel(p)
    return dict(case=case, model=m, pv=m.initial(), params=om.default_params(newton_tol=1e-10))


def _state(pv, mean):
    return {"sw": pv[0::3], "po": pv[1::3], "x": pv[2::3], "meaning": mean}


def run(state):
    kind = state["case"]["kind"]
    if kind == "steps":
        m, c = state["model"], state["res"]
        m.set_solution(c.pv0, c.mean0)
        rc, _, dts, _, _ = m.simulate(state["params"], state["case"]["steps"], state["params"].max_dt,
                                      keep_history=False)
        if rc != 0:
            raise RuntimeError("simulate returned %d" % rc)
        return dict(_state(*m.get_solution()), dts=dts)
    if kind == "iteration":
        m, s, case = state["model"], state["solver"], state["case"]
        m.set_solution(state["pv"], state["mean"])
        out = {}
        if case["host"]:
            J, r = m.linearize(DAY, iteration_index=0)
            out["jac"], out["res"] = J, r
            s.prepare(J, r)
        else:
            om.check(om.lib().omodels_linearizer_linearize_domain(m.h, DAY, 0), "linearize_domain")
            s.prepare()
        rc, x, _ = s.solve()
        if rc != 0:
            raise RuntimeError("solve returned %d" % rc)
        out["dsw"], out["dpo"], out["dx"] = x[0::3], x[1::3], x[2::3]
        m.newton_update(x, state["params"])
        out.update(_state(*m.get_solution()))
        if case["report"]:
            out["flows"], out["flores"] = m.flows()
            out["fields"] = m.output_fields()
        return out
    if kind == "serve":
        srv = state["server"]
        ids = [srv.submit(c, state["case"]["steps"], DAY) for c in state["requests"]]
        srv.run()
        out = []
        for i in ids:
            r = srv.result(i)
            if r["status"] != 0:
                raise RuntimeError("request %d: status %d" % (i, r["status"]))
            out.append(_state(r["pv"], r["mean"]))
        return out
    m = state["model"]
    m.set_solution(state["pv"])
    rc, _, dth, _, _ = m.simulate(state["params"], state["case"]["t_end"], 250.0, max_steps=100)
    if rc != 0:
        raise RuntimeError("lens simulate returned %d" % rc)
    pv = m.get_solution()
    return {"pw": pv[0::2], "sw": pv[1::2], "dts": dth}


# ---------------------------------------------------------------------------
def _newton_bytes(nx, ny, nz, order, precond, precision, its):
    """One Newton iteration: the state in and J, r out once; the matrix read
    and the preconditioner formed once; per BiCGStab iteration two operator
    applications (matrix, x, y), two preconditioner applications (their blocks
    and vectors) and the vector updates (each of p, r, x, v, y, z in and out)."""
    N = nx * ny * nz
    nnzb = N + 2 * ((nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1))
    s = 8 if precision == 0 else 4
    vec = 3 * s * N
    linearize = N * 69 + 24 * N + 72 * nnzb
    spmv = 9 * s * nnzb + 2 * vec
    if precond == 2:
        # two sweeps before and after, residual, transfers; coarser levels add 1/27 each
        prec = (4 * ((nnzb - N) * 9 * s + 72 * N + 3 * vec) + 9 * s * nnzb + 5 * vec) * 27 / 26
        setup = 72 * nnzb * 27 / 26 + 72 * N
    elif order == 1:
        prec = (nnzb - N) * 9 * s + 2 * 72 * N + 4 * vec
        setup = 72 * nnzb + 72 * N
    else:
        prec = 9 * s * (nnzb - N) + 72 * N + 3 * vec
        setup = 2 * 72 * nnzb
    flops = its * (4 * 18 * nnzb + 40 * 3 * N) + 100 * nnzb
    return linearize + setup + its * (2 * (spmv + prec) + 12 * vec), flops


def _its(order, precond, N):
    """Typical BiCGStab iterations per Newton iteration."""
    if precond == 2:
        return 7
    return max(4, int((25 if order == 0 else 31) * min(1.0, (N / 500e3) ** 0.25)))


def work(case):
    kind = case["kind"]
    if kind == "lens":
        n = case["nx"] * case["ny"]
        nnzb = 5 * n
        newton = 8 * case["t_end"] / 250.0          # Newton iterations, ten BiCGStab iterations each
        return {"bytes": newton * (32 * nnzb * 46 + 16 * n * 400), "flops": newton * (10 * 4 * 8 * nnzb)}
    if kind == "serve":
        N = case["requests"] * 0.5 * (case["cells_min"] + case["cells_max"])
        nz = 10
        nxy = math.sqrt(N / nz)
        b, f = _newton_bytes(nxy, nxy, nz, case["order"], 0, case["precision"],
                             _its(case["order"], 0, N / case["requests"]))
        return {"bytes": 8 * case["steps"] * b, "flops": 8 * case["steps"] * f}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    N = nx * ny * nz
    b, f = _newton_bytes(nx, ny, nz, case["order"], case["precond"], case["precision"],
                         _its(case["order"], case["precond"], N))
    if kind == "steps":
        return {"bytes": 9.0 * case["steps"] * b, "flops": 9.0 * case["steps"] * f}
    if case["report"]:
        b += 6 * N * 48 + 24 * N * 8
    return {"bytes": b, "flops": f}


def tolerance(case):
    """What the results leave open, measured on these cases by running them
    with the FP32 inner solve or another preconditioner in place of the
    case's own and taking about four times the largest difference.  A Newton
    run ends at its tolerance on the residual: pressures move by up to 2e-7,
    saturations by less, single cells by up to 4e-7 of the root mean square.
    A single Newton iteration's update is only as good as its linear solve
    (FP32 inner solve against FP64: 5e-6, single cells 6e-4; a cell on the
    bubble point may take the other gas meaning).  The lens run converges to
    1e-10: 4e-12, its step sizes the same."""
    if case["kind"] == "iteration":
        return {"rel": 2e-5, "max": 3e-3, "differ": 1e-4}
    if case["kind"] == "lens":
        return {"rel": 2e-11, "max": 2e-10}
    return {"rel": 1e-6, "max": 1e-5, "differ": 1e-4}


# ---------------------------------------------------------------------------
# The same equations in plain numpy (FP64, derivatives by complex step).
class _Tab:
    def __init__(self, x, y):
        self.x, self.y = np.asarray(x, float), np.asarray(y, float)
        self.s = np.diff(self.y) / np.diff(self.x)

    def __call__(self, v):
        i = np.clip(np.searchsorted(self.x, np.real(v), side="right") - 1, 0, len(self.s) - 1)
        return self.y[i] + self.s[i] * (v - self.x[i])


class _Plain:
    def __init__(self, c):
        s, self.c = c.spec, c
        self.shape = (s.nz, s.ny, s.nx)
        n, g = c.n_oil, c.n_gas
        oil, gas = c.oil.reshape(4, n), c.gas.reshape(3, g)
        self.rs, self.pb = _Tab(oil[0], oil[1]), _Tab(oil[1], oil[0])
        self.bo, self.muo = _Tab(oil[0], oil[2]), _Tab(oil[0], oil[3])
        self.bg, self.mug = _Tab(gas[0], gas[1]), _Tab(gas[0], gas[2])
        self.co, self.pref, self.cw, self.muw = c.consts[:4]
        self.rho = c.consts[4:7]
        self.V = s.dx * s.dy * s.dz
        h = (s.dz, s.dy, s.dx)
        k = [c.perm.reshape(3, *self.shape)[q] for q in (2, 1, 0)]
        self.half = [(self.V / h[a]) * k[a] / (0.5 * h[a]) for a in range(3)]
        z = s.dz * (np.arange(s.nz) + 0.5)
        self.z = np.broadcast_to(z[:, None, None], self.shape)

    def cell(self, x, mean):
        """phases water, oil, gas: mobility, 1/B, density; and p, Rs, saturations"""
        sw, p, y = x
        gas = mean == 0
        sg = np.where(gas, y, 0.0)
        S = (sw, 1.0 - sw - sg, sg)
        Rs = np.where(gas, self.rs(p), y)
        X = (p - self.pref) * self.cw
        pb = np.where(gas, p, self.pb(Rs))
        bo = self.bo(pb) * np.where(gas, 1.0, 1.0 + self.co * (p - pb))
        b = (1.0 + X * (1.0 + 0.5 * X), bo, self.bg(p))
        mu = (self.muw, self.muo(pb), self.mug(p))
        kr = [np.where(np.real(v) > 1.0, 1.0, np.where(np.real(v) < 0.0, 0.0, v)) for v in S]
        rho = (b[0] * self.rho[0], b[1] * (self.rho[1] + Rs * self.rho[2]), b[2] * self.rho[2])
        return dict(p=p, Rs=Rs, S=S, b=b, lam=[kr[a] / mu[a] for a in range(3)], rho=rho)

    def storage(self, q):
        phi = self.c.poro.reshape(self.shape)
        v = [q["S"][a] * q["b"][a] * phi for a in range(3)]
        return np.stack([v[1] * self.rho[1], v[0] * self.rho[0], (v[2] + q["Rs"] * v[1]) * self.rho[2]])

    def flux(self, own, oth, axis, up):
        """mass rates out of the cells `own` (slice) into their neighbours"""
        sl = [slice(None)] * 3
        so, sn = list(sl), list(sl)
        n = self.shape[axis]
        so[axis], sn[axis] = (slice(0, n - 1), slice(1, n)) if up else (slice(1, n), slice(0, n - 1))
        so, sn = tuple(so), tuple(sn)
        h = self.half[axis]
        T = 1.0 / (1.0 / h[so] + 1.0 / h[sn])
        dzg = (self.z[so] - self.z[sn]) * -9.81
        out = [0.0, 0.0, 0.0]
        for a in range(3):
            dp = oth["p"][sn] + 0.5 * (own["rho"][a][so] + oth["rho"][a][sn]) * dzg - own["p"][so]
            upin = (np.real(dp) < 0.0) | ((np.real(dp) == 0.0) & up)
            pick = lambda u, w: np.where(upin, u[so], w[sn])  # noqa: E731
            v = -T * dp * pick(own["lam"][a], oth["lam"][a]) * pick(own["b"][a], oth["b"][a])
            if a == 1:
                out[0] = out[0] + v * self.rho[1]
                out[2] = out[2] + v * pick(own["Rs"], oth["Rs"]) * self.rho[2]
            else:
                out[1 if a == 0 else 2] = out[1 if a == 0 else 2] + v * self.rho[a]
        return np.stack(out), so, sn

    def source(self, q):
        """mass rates into the cells"""
        s = np.zeros((3,) + self.shape, dtype=q["p"].dtype).reshape(3, -1)
        c = self.c
        for I, t, a, b in zip(c.src_cell, c.src_type, c.src_a, c.src_b):
            if t == 0:
                s[1, I] += a
                continue
            at = lambda v: np.ravel(v)[I]  # noqa: E731
            drive = at(q["p"]) - b
            if drive.real <= 0.0:
                continue
            v = [-a * at(q["lam"][f]) * at(q["b"][f]) * drive for f in range(3)]
            s[0, I] += v[1] * self.rho[1]
            s[1, I] += v[0] * self.rho[0]
            s[2, I] += (v[2] + at(q["Rs"]) * v[1]) * self.rho[2]
        return s.reshape((3,) + self.shape)

    def system(self, pv, mean, st1, dt):
        """residual [3N] and the blocks by slot (-z, -y, -x, own, +x, +y, +z), [7][N][3][3]"""
        N = self.c.N
        x = [pv[k::3].reshape(self.shape) for k in range(3)]
        mean = mean.reshape(self.shape)
        q0 = self.cell(x, mean)
        st = self.storage(q0)
        if st1 is None:
            st1 = st
        r = (st - st1) * (self.V / dt) - self.source(q0)
        for axis in range(3):
            for up in (True, False):
                f, so, _ = self.flux(q0, q0, axis, up)
                r[(slice(None),) + so] += f
        B = np.zeros((7, 3, 3) + self.shape)
        h = 1e-30
        for k in range(3):
            q = self.cell([x[m] + (1j * h if m == k else 0j) for m in range(3)], mean)
            B[3, :, k] += np.imag(self.storage(q)) / h * (self.V / dt) - np.imag(self.source(q)) / h
            for axis in range(3):
                for up in (True, False):
                    f, so, sn = self.flux(q, q0, axis, up)
                    d = np.imag(f) / h
                    B[(3, slice(None), k) + so] += d
                    # the neighbour's row, whose column for this cell lies the other way
                    B[(axis if up else 6 - axis, slice(None), k) + sn] -= d
        return r.reshape(3, N).T.ravel(), np.moveaxis(B.reshape(7, 3, 3, N), 3, 1), st

    def present(self):
        nz, ny, nx = self.shape
        k, j, i = np.indices(self.shape).reshape(3, -1)
        return np.stack([k > 0, j > 0, i > 0, k >= 0, i + 1 < nx, j + 1 < ny, k + 1 < nz])

    def bcrs(self, B):
        """the blocks row by row with sorted columns"""
        return np.moveaxis(B, 0, 1)[self.present().T].ravel()

    def dense(self, B):
        nz, ny, nx = self.shape
        N = self.c.N
        A = np.zeros((N, 3, N, 3))
        row = np.arange(N)
        has = self.present()
        for d, off in enumerate((-nx * ny, -nx, -1, 0, 1, nx, nx * ny)):
            R = row[has[d]]
            A[R, :, R + off, :] = B[d][R]
        return A.reshape(3 * N, 3 * N)

    def step(self, pv, mean, dt):
        """one implicit step by Newton's method with a dense solver"""
        st1 = None
        for it in range(40):
            r, B, st = self.system(pv, mean, st1, dt)
            st1 = st if st1 is None else st1
            if np.max(np.abs(r)) < 1e-11:
                break
            A = self.dense(B)
            w = np.tile([1.0, 1e7, 10.0], self.c.N)
            d = w * np.linalg.solve(A * w, r)
            d[0::3] = np.clip(d[0::3], -0.2, 0.2)
            pv = pv - d
            p, y = pv[1::3], pv[2::3]
            rs = self.rs(p)
            gas = mean == 0
            gone, come = gas & (y < 0.0), ~gas & (y > rs)
            y = np.where(gone, rs, np.where(come, 0.0, y))
            mean = np.where(gone, 1, np.where(come, 0, mean)).astype(np.uint8)
            pv[2::3] = y
            if it > 4 and np.max(np.abs(d / w)) < 1e-13:
                break
        return pv, mean


def exact(case, seed):
    if case["kind"] == "iteration":
        if not case["host"]:
            return None
        c = _reservoir(case, seed)
        m = _Plain(c)
        r, B, _ = m.system(*_disturbed(c, seed + 1), None, DAY)
        none = dict.fromkeys(("dsw", "dpo", "dx", "sw", "po", "x", "meaning"))
        if case["report"]:
            none.update(flows=None, flores=None, fields=None)
        return dict(none, jac=m.bcrs(B), res=r)
    if case["kind"] == "steps" and not case.get("terms") and case["nx"] * case["ny"] * case["nz"] <= 800:
        c = _reservoir(case, seed)
        m = _Plain(c)
        pv, mean = c.pv0.copy(), c.mean0.copy()
        for _ in range(case["steps"]):
            pv, mean = m.step(pv, mean, DAY)
        return dict(_state(pv, mean), dts=np.full(case["steps"], DAY))
    return None

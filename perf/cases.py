"""The work that users of this package have it do, as cases for timing.

A case names its kind:
  rhs    one right-hand side k = dt M^-1 R(u) on the caller's device buffers
         (Solver.rhs_device_noalloc): the call of a program with its own time
         integrator;
  run    one solve: project the initial condition, take `steps` steps (or
         integrate to `t_end`), read the state back;
  batch  a ragged batch of solves advanced together, every state read back;
  serve  a burst of requests to the solve server, every state read back.

Meshes are the package's seeded jittered periodic squares (nx x nx squares,
2 nx^2 triangles), or for the supersonic vortex a quarter ring between the
arcs r = 1 and r = 1.384, numbered row by row, with walls, inflow and outflow.
Single-precision solves hand their results on as float32.
"""
import math
from fractions import Fraction

import numpy as np
import torch

import dgcuda_amd as dg

CFL = 0.3
_stream = None


def listed():
    return [
        # One right-hand side of the smallest configuration (linear advection,
        # p = 1, 32 x 32 squares): nothing but launches and latency.
        dict(name="rhs_adv_p1_2k_fp64", kind="rhs", physics="advection", p=1, nx=32, precision="fp64"),
        # The same call for a user's own integrator on the isentropic-vortex
        # configuration, with an element count that divides by no tile.
        dict(name="rhs_euler_p2_32k_fp64", kind="rhs", physics="euler", p=2, nx=127, precision="fp64"),
        # The largest right-hand side the call's fixed scratch takes.
        dict(name="rhs_euler_p4_131k_fp32", kind="rhs", physics="euler", p=4, nx=256, precision="fp32"),
        # The advection configuration as a whole solve (a pulse, a fifth of a
        # period): about 250 steps of a problem far smaller than the chip.
        dict(name="run_adv_p1_2k_fp64", kind="run", physics="advection", p=1, nx=32, precision="fp64", scheme="rk4",
             t_end=2.0, steps=0),
        # The isentropic-vortex configuration (128 x 128 squares, p = 2), in
        # the two precisions it is run in.
        dict(name="run_euler_p2_32k_fp64", kind="run", physics="euler", p=2, nx=128, precision="fp64", scheme="rk4",
             t_end=0.0, steps=200),
        dict(name="run_euler_p2_32k_fp32", kind="run", physics="euler", p=2, nx=128, precision="fp32", scheme="rk4",
             t_end=0.0, steps=200),
        # The headline solve: p = 4 on 524,288 triangles, 200 steps.
        dict(name="run_euler_p4_524k_fp32", kind="run", physics="euler", p=4, nx=512, precision="fp32", scheme="rk4",
             t_end=0.0, steps=200),
        # A large solve at low order, the top of the request sizes (500k).
        dict(name="run_euler_p1_500k_fp32", kind="run", physics="euler", p=1, nx=500, precision="fp32", scheme="rk4",
             t_end=0.0, steps=200),
        # A large solve in double precision at the order between the two.
        dict(name="run_euler_p3_131k_fp64", kind="run", physics="euler", p=3, nx=256, precision="fp64", scheme="rk4",
             t_end=0.0, steps=100),
        # The reference program's problem: walls, inflow and outflow, a mesh
        # in its file's own numbering, the two-stage scheme.
        dict(name="run_supersonic_p2_8k_fp64", kind="run", physics="supersonic", p=2, nx=37, precision="fp64",
             scheme="rk2", t_end=0.0, steps=200),
        # A ragged batch, half advection pulses and half vortices, p = 1..4.
        dict(name="batch_32_fp32", kind="batch", solves=32, kmin=500, kmax=100000, steps=40, precision="fp32"),
        # A burst of small requests to the server.
        dict(name="serve_24_fp32", kind="serve", requests=24, kmin=1000, kmax=8000, precision="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    precision = rng.choice(["fp64", "fp32"])
    kind = rng.choice(["rhs", "rhs", "run", "run", "run", "batch"])
    if kind == "batch":
        return dict(kind="batch", solves=rng.randint(2, 32), kmin=500, kmax=_log_int(rng, 2000, 60000),
                    steps=rng.randint(5, 40), precision=precision)
    physics = rng.choice(["euler", "euler", "advection"])
    p = rng.randint(1, 4)
    if kind == "rhs":
        # double precision holds 16 mode slots per variable: half the triangles
        top = 256 if precision == "fp32" else 181
        return dict(kind="rhs", physics=physics, p=p, nx=_log_int(rng, 20, top), precision=precision)
    if rng.random() < 0.2:
        return dict(kind="run", physics="supersonic", p=rng.randint(1, 4), nx=_log_int(rng, 12, 60),
                    precision="fp64", scheme="rk2", t_end=0.0, steps=rng.randint(20, 200))
    return dict(kind="run", physics=physics, p=p, nx=_log_int(rng, 16, 320), precision=precision,
                scheme=rng.choice(["rk4", "rk4", "rk2"]), t_end=0.0, steps=rng.randint(20, 200))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _size(case):
    """(rows, columns) of squares of the case's mesh."""
    if case["physics"] == "supersonic":
        return case["nx"], 3 * case["nx"]
    return case["nx"], case["nx"]


def _ring(nr, nt, rng):
    """A quarter ring of nr x nt squares split into triangles, interior
    vertices jittered, in read_mesh's arrays."""
    r = 1.0 + 0.384 * np.arange(nr + 1) / nr
    th = 0.5 * np.pi * np.arange(nt + 1) / nt
    R, T = np.meshgrid(r, th, indexing="ij")
    R, T = R.copy(), T.copy()
    R[1:-1, 1:-1] += rng.uniform(-0.1, 0.1, (nr - 1, nt - 1)) * (0.384 / nr)
    T[1:-1, 1:-1] += rng.uniform(-0.1, 0.1, (nr - 1, nt - 1)) * (0.5 * np.pi / nt)
    X, Y = (R * np.cos(T)).ravel(), (R * np.sin(T)).ravel()
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nr), np.arange(nt), indexing="ij"))
    a = i * (nt + 1) + j
    b, c, d = a + nt + 1, a + nt + 2, a + 1
    tri = np.empty((2 * nr * nt, 3), np.int64)
    tri[0::2] = np.stack([a, b, c], 1)
    tri[1::2] = np.stack([a, c, d], 1)
    K = len(tri)
    ends = np.stack([tri, np.roll(tri, -1, 1)], 2).reshape(-1, 2)  # face f of element e at 3 e + f
    key = np.sort(ends, 1)
    _, first, side = np.unique(key[:, 0] * X.size + key[:, 1], return_index=True, return_inverse=True)
    S = len(first)
    left, lf = first // 3, first % 3
    other = np.full(S, -1)
    late = np.setdiff1d(np.arange(3 * K), first)
    other[side[late]] = late
    p0, p1 = ends[first, 0], ends[first, 1]
    t0, t1 = p0 % (nt + 1), p1 % (nt + 1)
    kind = np.where((t0 == 0) & (t1 == 0), -2, np.where((t0 == nt) & (t1 == nt), -3, -1))
    right = np.where(other >= 0, other // 3, kind)
    rf = np.where(other >= 0, other % 3, 0)
    V = np.stack([X[tri[:, 0]], Y[tri[:, 0]], X[tri[:, 1]], Y[tri[:, 1]], X[tri[:, 2]], Y[tri[:, 2]]])
    es = side.reshape(K, 3).T
    return V, es, np.stack([X[p0], Y[p0], X[p1], Y[p1]]), np.stack([left, right, lf, rf])


def _problem(physics, rng, L=10.0, speed=None):
    """(problem, its parameters) drawn by the generator."""
    if physics == "supersonic":
        par = dict(physics=physics, mach=float(rng.uniform(2.1, 2.4)))
        return dg.supersonic_vortex(mach=par["mach"]), par
    if physics == "advection":
        ang = rng.uniform(0, 2 * math.pi)
        s = math.sqrt(2.0) if speed is None else speed
        par = dict(physics=physics, a=(s * math.cos(ang), s * math.sin(ang)),
                   center=(float(rng.uniform(0, L)), float(rng.uniform(0, L))), k=1.0)
        return dg.advection_gaussian(a=par["a"], center=par["center"], k=par["k"]), par
    par = dict(physics=physics, vortices=tuple((float(rng.uniform(2, 5)), float(rng.uniform(0, L)),
                                                float(rng.uniform(0, L))) for _ in range(3)))
    return dg.euler_vortex(par["vortices"]), par


def _mesh(case, rng):
    nr, nt = _size(case)
    if case["physics"] == "supersonic":
        return dg.Mesh.from_arrays(*_ring(nr, nt, rng))
    return dg.Mesh.periodic_jittered(nr, nt, 0.0, 10.0, 0.0, 10.0, 0.1, int(rng.integers(1, 2**31)))


def _batch(case, seed):
    """[(mesh, problem, parameters, p)] of a ragged batch."""
    rng = np.random.default_rng(seed)
    shape = np.random.default_rng(7)  # sizes and orders belong to the case
    out = []
    for i in range(case["solves"]):
        nx = max(2, int(round(math.sqrt(math.exp(shape.uniform(math.log(case["kmin"]), math.log(case["kmax"]))) / 2))))
        p = int(shape.integers(1, 5))
        m = dg.Mesh.periodic_jittered(nx, nx, 0.0, 10.0, 0.0, 10.0, 0.1, int(rng.integers(1, 2**31)))
        prob, par = _problem("advection" if i % 2 == 0 else "euler", rng, speed=float(rng.uniform(0.1, 1.0)))
        out.append((m, prob, par, p))
    return out


def _requests(case, seed):
    """[(nx, p, t_end, mesh seed, problem, parameters)] of a burst."""
    rng = np.random.default_rng(seed)
    shape = np.random.default_rng(11)
    out = []
    for _ in range(case["requests"]):
        nx = int(round(math.sqrt(math.exp(shape.uniform(math.log(case["kmin"]), math.log(case["kmax"]))) / 2)))
        p, te = int(shape.integers(1, 4)), float(shape.uniform(0.05, 0.2))
        prob, par = _problem("euler", rng)
        out.append((nx, p, te, int(rng.integers(1, 2**31)), prob, par))
    return out


def _precision(case):
    return dg.DG_FP64 if case["precision"] == "fp64" else dg.DG_FP32


def _rhs_input(mesh, p, par, rng):
    """A state in the caller's layout: the initial condition plus a small
    perturbation of every mode, as in the midst of a run."""
    u = _Exact(mesh, p, par, "cpu" if mesh.num_elem < 5000 else None).project()
    amp = 1e-2 * min(1.0, 6.0 / u.shape[1]) * (u.abs().amax(dim=(1, 2), keepdim=True) + 1e-3)
    gen = torch.Generator().manual_seed(int(rng.integers(1, 2**31)))
    return u + amp * torch.randn(u.shape, generator=gen, dtype=torch.float64).to(u.device)


def _on_stream():
    """The one stream of this program's own integrators: their calls share
    the package's scratch and must not overlap."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _rhs_parts(case, seed):
    rng = np.random.default_rng(seed)
    mesh = _mesh(case, rng)
    prob, par = _problem(case["physics"], rng)
    return mesh, prob, par, _rhs_input(mesh, case["p"], par, rng)


RHS_DT = 1e-3


def prepare(case, seed):
    kind = case["kind"]
    if kind == "rhs":
        mesh, prob, _, u = _rhs_parts(case, seed)
        u = u.cuda().contiguous()
        solver = dg.Solver(mesh, prob, case["p"], _precision(case))
        k = torch.zeros_like(u)
        torch.cuda.synchronize()
        return dict(case=case, solver=solver, u=u, k=k, stream=_on_stream())
    if kind == "run":
        rng = np.random.default_rng(seed)
        mesh = _mesh(case, rng)
        prob, _ = _problem(case["physics"], rng)
        return dict(case=case, solver=dg.Solver(mesh, prob, case["p"], _precision(case)))
    if kind == "batch":
        b = dg.Batch(_precision(case))
        for m, prob, _, p in _batch(case, seed):
            b.add(m, prob, p, 1e30)
        return dict(case=case, batch=b)
    sv = dg.Server(_precision(case))
    sv.keep_states(True)
    return dict(case=case, server=sv, requests=_requests(case, seed))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _result(case, c):
    """A state as a user of the precision keeps it."""
    c = torch.from_numpy(c)
    return c if case["precision"] == "fp64" else c.float()


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "rhs":
        st = state["stream"]
        state["solver"].rhs_device_noalloc(state["u"].data_ptr(), state["k"].data_ptr(), RHS_DT, st.cuda_stream)
        if case["precision"] == "fp64":
            return state["k"]
        with torch.cuda.stream(st):
            return state["k"].float()
    if kind == "run":
        s = state["solver"]
        scheme = dg.DG_RK4 if case["scheme"] == "rk4" else dg.DG_RK2
        s.project_ic()
        if case["t_end"] > 0:
            s.integrate(case["t_end"], CFL, scheme)
        else:
            s.run_steps(case["steps"], CFL, scheme)
        return _result(case, s.get_state())
    if kind == "batch":
        b = state["batch"]
        b.project_ic()
        b.run_steps(case["steps"], CFL)
        return [_result(case, b.get_state(i)) for i in range(case["solves"])]
    sv = state["server"]
    ids = [sv.submit(dg.request(nx, p, te, prob, mesh_seed=ms)) for nx, p, te, ms, prob, _ in state["requests"]]
    sv.drain()
    sv.poll(len(ids))
    return [_result(case, sv.get_state(i, (4, dg.n_modes(r[1]), 2 * r[0] * r[0])))
            for i, r in zip(ids, state["requests"])]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
_NQ = {1: 3, 2: 6, 3: 12, 4: 16}


def _stage_flops(K, N, p):
    """Multiply-adds (two each) of the contractions and the fluxes of one
    right-hand side: volume interpolation and projection, each side's two
    traces and one flux, the surface projection."""
    NP, NQ, n1 = (p + 1) * (p + 2) // 2, _NQ[p], p + 1
    flux = 2.0 if N == 1 else 35.0
    return K * (2.0 * N * NP * (3 * NQ + 2 * 3 * n1) + flux * (NQ + 1.5 * n1))


def _solve_work(K, N, p, s, steps, arrays, stages):
    """A run: per step the state arrays its scheme reads and writes and per
    stage the geometry (7 values and 3 neighbours an element: its map, its
    inverse mass, its sides' share), the state written once at first and
    handed over as 64 bits at last."""
    NP = (p + 1) * (p + 2) // 2
    state = float(K) * N * NP
    per_step = arrays * state * s + stages * K * (7.0 * s + 12.0)
    return dict(bytes=steps * per_step + state * (2 * s + 8), flops=steps * stages * _stage_flops(K, N, p))


def _steps_of(case):
    if case["steps"]:
        return case["steps"]
    # cfl * r / (2p+1) / |a| with the jittered mesh's smallest inscribed circle
    h = 10.0 / case["nx"]
    return max(1, int(case["t_end"] / (CFL * 0.45 * h / (2 * case["p"] + 1) / math.sqrt(2.0))))


def work(case):
    kind = case["kind"]
    s = 8 if case["precision"] == "fp64" else 4
    if kind in ("rhs", "run"):
        nr, nt = _size(case)
        K, N, p = 2 * nr * nt, 1 if case["physics"] == "advection" else 4, case["p"]
        if kind == "rhs":
            NP = (p + 1) * (p + 2) // 2
            return dict(bytes=K * (16.0 * N * NP + 7.0 * s + 12.0), flops=_stage_flops(K, N, p))
        arrays, stages = (12, 4) if case["scheme"] == "rk4" else (5, 2)
        return _solve_work(K, N, p, s, _steps_of(case), arrays, stages)
    total = dict(bytes=0.0, flops=0.0)
    if kind == "batch":
        shape = np.random.default_rng(7)
        each = []
        for i in range(case["solves"]):
            K = math.exp(shape.uniform(math.log(case["kmin"]), math.log(case["kmax"])))
            each.append((K, 1 if i % 2 == 0 else 4, int(shape.integers(1, 5)), case["steps"]))
    else:
        shape = np.random.default_rng(11)
        each = []
        for _ in range(case["requests"]):
            K = math.exp(shape.uniform(math.log(case["kmin"]), math.log(case["kmax"])))
            p, te = int(shape.integers(1, 4)), float(shape.uniform(0.05, 0.2))
            h = 10.0 / math.sqrt(K / 2)
            each.append((K, 4, p, max(1, int(te / (CFL * 0.45 * h / (2 * p + 1) / 3.0)))))
    for K, N, p, steps in each:
        w = _solve_work(K, N, p, s, steps, 12, 4)
        total = dict(bytes=total["bytes"] + w["bytes"], flops=total["flops"] + w["flops"])
    return total


# ---------------------------------------------------------------------------
# the same numbers from plain torch in 64 bits
# ---------------------------------------------------------------------------
def _exponents(p):
    return [(d - b, b) for d in range(p + 1) for b in range(d + 1)]


def _basis(p):
    """Coefficients [mode][monomial] of the orthonormal basis on the triangle
    (0,0), (1,0), (0,1): Gram-Schmidt of 1, r, s, r^2, rs, s^2, ... with the
    exact moments a! b! / (a + b + 2)!, each mode positive in its last
    monomial (odd-signed ones as the published tables have them)."""
    ex = _exponents(p)
    f = math.factorial

    def dot(u, v):
        return sum((cu * cv * Fraction(f(a + c) * f(b + d), f(a + b + c + d + 2))
                    for cu, (a, b) in zip(u, ex) if cu for cv, (c, d) in zip(v, ex) if cv), Fraction(0))

    rows, out = [], []
    for k in range(len(ex)):
        v = [Fraction(int(i == k)) for i in range(len(ex))]
        for w in rows:
            h = dot(w, v) / dot(w, w)
            v = [x - h * y for x, y in zip(v, w)]
        rows.append(v)
        out.append([float(x) / math.sqrt(float(dot(v, v))) for x in v])
    return np.array(out)


def _volume_rule(p):
    """Symmetric triangle rules of degree 2p (3, 6, 12 and 16 points; Strang
    and Fix, Dunavant): points and weights, the weights summing to 1/2."""
    orbit3 = {1: [(1 / 6, 1 / 3)],
              2: [(0.445948490915965, 0.223381589678011), (0.091576213509771, 0.109951743655322)],
              3: [(0.249286745170910, 0.116786275726379), (0.063089014491502, 0.050844906370207)],
              4: [(0.459292588292723, 0.095091634267285), (0.170569307751760, 0.103217370534718),
                  (0.050547228317031, 0.032458497623198)]}[p]
    orbit6 = {3: [(0.310352451033784, 0.053145049844817, 0.082851075618374)],
              4: [(0.263112829634638, 0.008394777409958, 0.027230314174435)]}.get(p, [])
    pts = [(1 / 3, 1 / 3, 0.144315607677787)] if p == 4 else []
    for a, w in orbit3:
        b = 1 - 2 * a
        pts += [(a, a, w), (a, b, w), (b, a, w)]
    for a, b, w in orbit6:
        c = 1 - a - b
        pts += [(x, y, w) for x, y in ((a, b), (b, a), (a, c), (c, a), (b, c), (c, b))]
    pts = np.array(pts)
    return pts[:, 0], pts[:, 1], pts[:, 2] / 2


class _Exact:
    """Modal DG on the mesh's arrays in 64 bits, by dense torch products."""

    def __init__(self, mesh, p, par, device=None):
        self.dev = device or ("cuda" if torch.cuda.is_available() else "cpu")
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        self.p, self.par = p, par
        self.N = 1 if par["physics"] == "advection" else 4
        C, ex = _basis(p), _exponents(p)
        self.NP = len(ex)

        def phi(r, s, dr=0, ds=0):
            cols = []
            for a, b in ex:
                fa = {0: 1, 1: a}[dr]
                fb = {0: 1, 1: b}[ds]
                cols.append(fa * fb * r ** max(a - dr, 0) * s ** max(b - ds, 0))
            return C @ np.array(cols)

        r, s, w = _volume_rule(p)
        self.r, self.s, self.w = r, s, w
        self.B, self.Gr, self.Gs = t(phi(r, s)), t(phi(r, s, dr=1) * w), t(phi(r, s, ds=1) * w)
        x, self.w1 = np.polynomial.legendre.leggauss(p + 1)
        self.n1 = p + 1
        fr = [(0.5 + 0.5 * x, 0 * x), ((1 - x) / 2, (1 + x) / 2), (0 * x, (0.5 + 0.5 * x)[::-1])]
        self.face_rs = fr
        self.S = torch.stack([t(phi(a, b)) for a, b in fr])  # [3][NP][n1]
        self.w1 = t(self.w1)
        V, es, sd, si = mesh.arrays()
        self.period = mesh.period
        self.K = V.shape[1]
        x1, y1, x2, y2, x3, y3 = V
        self.V = V
        self.xr, self.yr, self.xs, self.ys = t(x2 - x1), t(y2 - y1), t(x3 - x1), t(y3 - y1)
        self.J = self.xr * self.ys - self.xs * self.yr
        a, b, c = np.hypot(x1 - x2, y1 - y2), np.hypot(x2 - x3, y2 - y3), np.hypot(x1 - x3, y1 - y3)
        h = 0.5 * (a + b + c)
        self.min_r = float((2 * np.sqrt(h * (h - a) * (h - b) * (h - c)) / h).min())
        left, right, lf, rf = si
        ln = np.hypot(sd[2] - sd[0], sd[3] - sd[1])
        nx, ny = -(sd[3] - sd[1]) / ln, (sd[2] - sd[0]) / ln
        opp = np.array([2, 0, 1])[lf]  # the left element's vertex off the side
        P = V.reshape(3, 2, -1)
        e0, e1 = P[lf, :, left], P[(lf + 1) % 3, :, left]
        flip = (nx * (P[opp, 0, left] - e0[:, 0] / 2 - e1[:, 0] / 2) +
                ny * (P[opp, 1, left] - e0[:, 1] / 2 - e1[:, 1] / 2)) > 0
        nx, ny = np.where(flip, -nx, nx), np.where(flip, -ny, ny)
        self.left, self.lf, self.rf = t(left.astype(np.int64)), t(lf.astype(np.int64)), t(rf.astype(np.int64))
        self.inner = t(right >= 0)
        self.right = t(np.where(right >= 0, right, left).astype(np.int64))
        self.len, self.nx, self.ny = t(ln), t(nx), t(ny)
        es = es.astype(np.int64)
        self.es = t(es)
        mine = (left[es] == np.arange(self.K)) & (lf[es] == np.arange(3)[:, None])
        self.is_left = t(mine)
        bs = np.nonzero(right < 0)[0]
        self.bs = t(bs)
        if len(bs):
            # ghost data at the boundary sides' points (left element's face)
            fx = np.empty((len(bs), self.n1))
            fy = np.empty((len(bs), self.n1))
            for f in range(3):
                q = lf[bs] == f
                a, b = fr[f]
                o = left[bs][q]
                fx[q] = x2[o][:, None] * a + x3[o][:, None] * b + x1[o][:, None] * (1 - a - b)
                fy[q] = y2[o][:, None] * a + y3[o][:, None] * b + y1[o][:, None] * (1 - a - b)
            self.wall = t(right[bs] == -1)
            d = np.hypot(fx, fy)
            self.wx, self.wy = t(fx / d), t(fy / d)
            self.ghost = t(self.initial(fx, fy))  # [4][side][point]

    def initial(self, x, y):
        par = self.par
        if par["physics"] == "supersonic":
            r2, M, g = x * x + y * y, par["mach"], 1.4
            r = np.sqrt(r2)
            rho = (1 + 1.0125 * (1 - 1 / r2)) ** 2.5
            th = np.arctan(y / x)
            pr = rho**g / g
            return np.stack([rho, rho * np.sin(th) * M / r, -rho * np.cos(th) * M / r,
                             0.5 * rho * M * M / r2 + pr / (g - 1)])
        wrap = lambda d, L: d - L * np.rint(d / L)  # noqa: E731
        Lx, Ly = self.period
        if par["physics"] == "advection":
            dx, dy = wrap(x - par["center"][0], Lx), wrap(y - par["center"][1], Ly)
            return np.exp(-par["k"] * (dx * dx + dy * dy))[None]
        g = 1.4
        u, v, T = np.ones_like(x), np.ones_like(x), np.ones_like(x)
        for b, xc, yc in par["vortices"]:
            dx, dy = wrap(x - xc, Lx), wrap(y - yc, Ly)
            e = np.exp(0.5 * (1 - dx * dx - dy * dy))
            u -= b / (2 * np.pi) * dy * e
            v += b / (2 * np.pi) * dx * e
            T -= (g - 1) * b * b / (8 * g * np.pi**2) * e * e
        rho = T ** (1 / (g - 1))
        return np.stack([rho, rho * u, rho * v, rho**g / (g - 1) + 0.5 * rho * (u * u + v * v)])

    def project(self):
        x1, y1, x2, y2, x3, y3 = (v[:, None] for v in self.V)
        q = 1 - self.r - self.s
        U = self.initial(x2 * self.r + x3 * self.s + x1 * q, y2 * self.r + y3 * self.s + y1 * q)  # [N][K][q]
        U = torch.as_tensor(U * self.w, device=self.dev)
        return (U @ self.B.T).transpose(1, 2).contiguous()  # [N][NP][K]

    def flux(self, U):
        """Cartesian fluxes of states U[N] (any trailing shape)."""
        if self.N == 1:
            return self.par["a"][0] * U, self.par["a"][1] * U
        rho, ru, rv, E = U
        u, v = ru / rho, rv / rho
        pr = 0.4 * (E - 0.5 * (ru * u + rv * v))
        return torch.stack([ru, ru * u + pr, ru * v, u * (E + pr)]), torch.stack([rv, rv * u, rv * v + pr, v * (E + pr)])

    def speed(self, U, nx, ny):
        if self.N == 1:
            return (self.par["a"][0] * nx + self.par["a"][1] * ny).abs().expand(U.shape[1:])
        rho, ru, rv, E = U
        pr = 0.4 * (E - 0.5 * (ru * ru + rv * rv) / rho)
        return ((ru * nx + rv * ny) / rho).abs() + torch.sqrt(1.4 * pr / rho)

    def rhs(self, c):
        """M^-1 R of c[N][NP][K]."""
        ct = c.transpose(1, 2)  # [N][K][NP]
        fx, fy = self.flux((ct @ self.B))
        col = lambda a: a[:, None]  # noqa: E731
        R = (fx * col(self.ys) - fy * col(self.xs)) @ self.Gr.T + (fy * col(self.xr) - fx * col(self.yr)) @ self.Gs.T
        del fx, fy
        T = torch.stack([ct @ self.S[f] for f in range(3)])  # [3][N][K][n1]
        UL = T[self.lf, :, self.left].permute(1, 0, 2)  # [N][side][n1]
        UR = T[self.rf, :, self.right].permute(1, 0, 2).flip(2)
        del T
        if len(self.bs):
            UR = UR.clone()
            L = UL[:, self.bs]
            tg = L[1] * self.wy - L[2] * self.wx
            refl = torch.stack([L[0], tg * self.wy, -tg * self.wx, L[3]])
            UR[:, self.bs] = torch.where(col(self.wall), refl, self.ghost)
        nx, ny = col(self.nx), col(self.ny)
        fxl, fyl = self.flux(UL)
        fxr, fyr = self.flux(UR)
        lam = torch.maximum(self.speed(UL, nx, ny), self.speed(UR, nx, ny))
        G = 0.5 * ((fxl + fxr) * nx + (fyl + fyr) * ny + lam * (UL - UR)) * self.w1 * (col(self.len) / 2)
        del UL, UR, fxl, fyl, fxr, fyr, lam
        for f in range(3):
            own = self.is_left[f]
            g = G[:, self.es[f]]  # [N][K][n1]
            g = torch.where(col(own), -g, g.flip(2))
            R = R + g @ self.S[f].T
        return R.transpose(1, 2) / self.J

    def dt(self, c):
        U = c[:, 0] * math.sqrt(2.0)
        if self.N == 1:
            lam = math.hypot(*self.par["a"])
        else:
            m = torch.sqrt(U[1] ** 2 + U[2] ** 2)
            pr = 0.4 * (U[3] - 0.5 * m * m / U[0])
            lam = float((m / U[0] + torch.sqrt(1.4 * pr / U[0])).max())
        return CFL * self.min_r / lam / (2 * self.p + 1)

    def step(self, c, dt, scheme):
        k1 = dt * self.rhs(c)
        k2 = dt * self.rhs(c + 0.5 * k1)
        if scheme == "rk2":
            return c + k2
        k3 = dt * self.rhs(c + 0.5 * k2)
        k4 = dt * self.rhs(c + k3)
        return c + (k1 + 2 * k2 + 2 * k3 + k4) / 6

    def run(self, scheme, steps=0, t_end=0.0):
        c, t, n = self.project(), 0.0, 0
        while (n < steps) if steps else (t < t_end):
            dt = self.dt(c)
            if not steps and t + dt > t_end:
                dt, t = t_end - t, t_end
            else:
                t += dt
            c = self.step(c, dt, scheme)
            n += 1
        return c.contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "rhs":
        mesh, _, par, u = _rhs_parts(case, seed)
        e = _Exact(mesh, case["p"], par)
        return (RHS_DT * e.rhs(u.to(e.dev))).contiguous()
    if kind == "run":
        nr, nt = _size(case)
        if 2.0 * nr * nt * (case["p"] + 1) ** 2 * case["steps"] > 3e9:
            return None  # minutes of 64-bit arithmetic
        rng = np.random.default_rng(seed)
        mesh = _mesh(case, rng)
        _, par = _problem(case["physics"], rng)
        return _Exact(mesh, case["p"], par).run(case["scheme"], case["steps"], case["t_end"])
    if kind == "batch":
        return [_Exact(m, p, par).run("rk4", case["steps"]) for m, _, par, p in _batch(case, seed)]
    out = []
    for nx, p, te, ms, _, par in _requests(case, seed):
        m = dg.Mesh.periodic_jittered(nx, nx, 0.0, 10.0, 0.0, 10.0, 0.1, ms)
        out.append(_Exact(m, p, par).run("rk4", t_end=te))
    return out

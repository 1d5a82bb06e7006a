"""What is timed: the work a user of this framework has it do.

A case is a plain dict; prepare() makes what a program holds before the call
(grids, bodies, start fields, a resident compat case), run() is one pass
through the public entry points.  Kinds:

compat_ad   the reference's ADsolver on a resident case: load u, v, a few
            ADsolver calls, fetch u, v (the reference's own program loop).
compat_ppe  the reference's PPESolver: load p, solve, fetch p.
flow        a whole simulation job on one grid, as the command-line driver
            runs it: create the case (classification, ghost cells, initial
            state), time steps, fetch u, v, p.  With "tuned" the launch
            shape is autotuned after the first step, as the headline
            benchmark does.
batch       a set of uneven requests served together: admit them into a
            batch, one step, autotune, the remaining steps, fetch every
            request's u, v, p.

The autotuner also picks the interval of the convergence checks from its
timings; run() pins the interval again, as a program does that wants the
same stop decisions in every run.
"""
import math

import numpy as np
import torch

import immerseflow_amd as iff
from immerseflow_amd import configs

PRECISION = {"fp64": iff.IF_FP64, "mixed": iff.IF_MIXED, "mixed_v32": iff.IF_MIXED_V32}
SOLVER = {"rbsor": iff.IF_PPE_RBSOR, "line": iff.IF_PPE_LINE}


def listed():
    return [
        # the reference's own deck (50 x 50 cells, Re 150, dt 0.001): the
        # smallest calls, where a pass is launches and waits
        dict(name="compat_ad_50", kind="compat_ad", nx=50, ny=50, lx=1.0, ly=1.0, dt=0.001, re=150.0, steps=10),
        dict(name="compat_poisson_50", kind="compat_ppe", nx=50, ny=50, lx=1.0, ly=1.0, dt=0.001, re=150.0),
        # the smallest serving request (64^2), mixed precision
        dict(name="request_64", kind="flow", grid="uniform", n=64, length=20.0, body="stars", bodies=2, re=300.0,
             dt=0.0, precision="mixed", solver="rbsor", omega=0.0, tol=1e-7, check=160, steps=40, tuned=False),
        # the plain FP64 method: cylinder in a 16 x 16 box, 256^2, Re 100
        dict(name="cylinder_256_fp64", kind="flow", grid="uniform", n=256, length=16.0, body="circle", bodies=1,
             re=100.0, dt=0.002, precision="fp64", solver="rbsor", omega=0.0, tol=1e-8, check=10, steps=20, tuned=False),
        # the deck's PPE_Solver 2 (zebra line SOR) on the same flow
        dict(name="cylinder_256_line", kind="flow", grid="uniform", n=256, length=16.0, body="circle", bodies=1,
             re=100.0, dt=0.002, precision="fp64", solver="line", omega=0.0, tol=1e-8, check=40, steps=6, tuned=False),
        # a moving body: iBlank, ghost cells and weights rebuilt every step
        dict(name="heaving_611", kind="flow", grid="uniform", n=611, length=20.0, body="heave", bodies=1, re=400.0,
             dt=0.0, precision="mixed", solver="rbsor", omega=0.0, tol=1e-7, check=160, steps=12, tuned=False),
        # a large serving request of ragged size, mixed precision
        dict(name="request_1948", kind="flow", grid="uniform", n=1948, length=20.0, body="stars", bodies=3, re=700.0,
             dt=0.0, precision="mixed", solver="rbsor", omega=0.0, tol=1e-7, check=160, steps=6, tuned=False),
        # one large case on a stretched grid, mixed and FP64
        dict(name="ellipse_2048_mixed", kind="flow", grid="stretched", n=2048, length=30.0, body="ellipse", bodies=1,
             re=300.0, dt=0.0025, precision="mixed", solver="rbsor", omega=1.998, tol=1e-6, check=480, steps=12,
             tuned=True),
        dict(name="ellipse_2048_fp64", kind="flow", grid="stretched", n=2048, length=30.0, body="ellipse", bodies=1,
             re=300.0, dt=0.0025, precision="fp64", solver="rbsor", omega=1.998, tol=1e-6, check=160, steps=4,
             tuned=False),
        # the headline: eight star bodies on 4096^2, mixed precision
        dict(name="stars_4096", kind="flow", grid="uniform", n=4096, length=20.0, body="stars", bodies=8, re=1000.0,
             dt=0.0, precision="mixed", solver="rbsor", omega=0.0, tol=1e-7, check=1000, steps=3, tuned=True),
        # many uneven cases at once (128^2 .. 1024^2 circles and ellipses)
        dict(name="batch_uneven", kind="batch", requests="uneven", mix=4, count=20, lo=128, hi=1024, precision="mixed",
             tol=1e-7, check=320, steps=10),
        # a serving mix (64^2 .. 2048^2: stars, one in five a heaving cylinder)
        dict(name="serving_mix", kind="batch", requests="serving", mix=5, count=16, lo=64, hi=2048, precision="mixed",
             tol=1e-7, check=160, steps=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    if pick < 0.12:
        nx, ny = _log_int(rng, 12, 180), _log_int(rng, 12, 180)
        return dict(kind="compat_ad", nx=nx, ny=ny, lx=1.0, ly=rng.choice([0.5, 1.0, 2.0]),
                    dt=rng.choice([0.0005, 0.001, 0.002]), re=rng.uniform(50.0, 300.0), steps=rng.randint(2, 20))
    if pick < 0.22:
        return dict(kind="compat_ppe", nx=_log_int(rng, 12, 72), ny=_log_int(rng, 12, 72), lx=1.0, ly=1.0, dt=0.001,
                    re=150.0)
    if pick < 0.40:   # FP64, uniform
        n = _log_int(rng, 64, 1100)
        return dict(kind="flow", grid="uniform", n=n, length=16.0, body=rng.choice(["circle", "ellipse"]), bodies=1,
                    re=rng.uniform(50.0, 500.0), dt=0.0, precision="fp64", solver="rbsor", omega=0.0, tol=1e-8,
                    check=rng.choice([10, 40, 160]), steps=max(2, min(20, 3000 // n)), tuned=False)
    if pick < 0.50:   # line SOR
        n = _log_int(rng, 64, 384)
        return dict(kind="flow", grid="uniform", n=n, length=16.0, body="circle", bodies=1, re=rng.uniform(50.0, 200.0),
                    dt=0.0, precision=rng.choice(["fp64", "mixed"]), solver="line", omega=0.0, tol=1e-7, check=40,
                    steps=3, tuned=False)
    if pick < 0.75:   # one serving request
        n = _log_int(rng, 64, 2048)
        return dict(kind="flow", grid="uniform", n=n, length=20.0, body=rng.choice(["stars", "stars", "stars", "heave"]),
                    bodies=rng.randint(1, 3), re=rng.uniform(100.0, 1000.0), dt=0.0,
                    precision=rng.choice(["mixed", "mixed", "mixed_v32"]), solver="rbsor", omega=0.0, tol=1e-7,
                    check=160, steps=max(3, min(40, 10000 // n)), tuned=rng.random() < 0.4)
    if pick < 0.86:   # stretched
        n = _log_int(rng, 1100, 2048)
        return dict(kind="flow", grid="stretched", n=n, length=30.0, body="ellipse", bodies=1,
                    re=rng.uniform(100.0, 400.0), dt=0.0025, precision="mixed", solver="rbsor", omega=1.998, tol=1e-6,
                    check=480, steps=6, tuned=rng.random() < 0.5)
    serving = rng.random() < 0.5
    return dict(kind="batch", requests="serving" if serving else "uneven", mix=rng.randint(10, 9999),
                count=rng.randint(3, 20),
                lo=64 if serving else 128, hi=1400 if serving else 1024,
                precision=rng.choice(["mixed", "mixed", "mixed_v32"]), tol=1e-7, check=rng.choice([160, 320]),
                steps=rng.randint(3, 8))


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _rng(seed, salt):
    r = configs.SplitMix64(1000003 * int(seed) + salt)
    r.next()
    return r


def _flow_input(case, seed):
    rng = _rng(seed, 17)
    n = case["n"]
    re = case["re"] * rng.uniform(0.95, 1.05)
    if case["grid"] == "stretched":
        cfg = configs.c2((n, n // 2))
        xf, yf = cfg["xf"], cfg["yf"]
        bodies = [iff.ellipse(15.0, 10.0, 0.5, 0.05, math.radians(rng.uniform(8.0, 12.0)))]
    else:
        length = case["length"]
        xf = configs.uniform_faces(n, length)
        yf = xf.copy()
        if case["body"] == "circle":
            bodies = [iff.circle(5.0 + rng.uniform(-0.2, 0.2), 8.0 + rng.uniform(-0.2, 0.2), 0.5)]
        elif case["body"] == "ellipse":
            bodies = [iff.ellipse(5.0, 8.0, 0.5, 0.5 / rng.uniform(1.0, 5.0), rng.uniform(0.0, math.pi))]
        elif case["body"] == "heave":
            bodies = [iff.heaving_circle(6.0 + rng.uniform(-0.2, 0.2), 10.0, 0.5, 0.5, 0.2)]
        else:
            bodies = configs.star_set(rng, case["bodies"], 2.0, 18.0)
    dt = case["dt"] if case["dt"] > 0 else (0.5 * case["length"] / n if n >= 4096
                                             else configs.stable_dt(case["length"] / n, re))
    return dict(xf=xf, yf=yf, bodies=bodies, re=re, dt=dt)


def _requests(case, seed):
    rng, sizes = _rng(seed, 29), _rng(case["mix"], 31)
    out = []
    # stratified in log size, so that every set has its small and large grids
    for k in range(case["count"]):
        t = (k + sizes.uniform()) / case["count"]
        n = int(round(math.exp(math.log(case["lo"]) + t * (math.log(case["hi"]) - math.log(case["lo"])))))
        if case["requests"] == "uneven":
            length, re = 16.0, rng.uniform(50.0, 500.0)
            if rng.uniform() < 0.5:
                bodies = [iff.circle(5.0, 8.0, 0.5)]
            else:
                bodies = [iff.ellipse(5.0, 8.0, 0.5, 0.5 / rng.uniform(1.0, 5.0), rng.uniform(0.0, math.pi))]
        else:
            length, re = 20.0, rng.uniform(100.0, 1000.0)
            if k % 5 == 2:
                bodies = [iff.heaving_circle(6.0, 10.0, 0.5, 0.5, 0.2)]
            else:
                bodies = configs.star_set(rng, 1 + int(rng.uniform() * 3), 2.0, 18.0)
        xf = configs.uniform_faces(n, length)
        out.append(dict(xf=xf, yf=xf.copy(), bodies=bodies, dt=configs.stable_dt(length / n, re), re=re))
    return out


def _compat_fields(case, seed):
    """(xf, yf, u, v, p): the reference's vortex at a seeded place; p linear,
    below the 100 that the west and south edges are held at."""
    rng = _rng(seed, 41)
    xf = np.linspace(0.0, case["lx"], case["nx"] + 1)
    yf = np.linspace(0.0, case["ly"], case["ny"] + 1)
    xc = np.concatenate(([-0.5 * xf[1]], 0.5 * (xf[:-1] + xf[1:]), [xf[-1] + 0.5 * (xf[-1] - xf[-2])]))
    yc = np.concatenate(([-0.5 * yf[1]], 0.5 * (yf[:-1] + yf[1:]), [yf[-1] + 0.5 * (yf[-1] - yf[-2])]))
    x, y = np.meshgrid(xc, yc)
    x0, y0, r0 = rng.uniform(0.3, 0.7) * case["lx"], rng.uniform(0.3, 0.7) * case["ly"], rng.uniform(0.08, 0.15)
    e = 0.25 * np.exp((1.0 - ((x - x0) ** 2 + (y - y0) ** 2) / r0 ** 2) / 2.0)
    u, v = 1.0 - (y - y0) * e, (x - x0) * e
    p = rng.uniform(5.0, 20.0) + rng.uniform(0.0, 20.0) * x / case["lx"] + rng.uniform(0.0, 20.0) * y / case["ly"]
    return xf, yf, u.ravel(), v.ravel(), p.ravel()


def prepare(case, seed):
    if case["kind"] in ("compat_ad", "compat_ppe"):
        xf, yf, u, v, p = _compat_fields(case, seed)
        c = iff.Case(xf, yf, mode=iff.IF_MODE_COMPAT, dt=case["dt"], re=case["re"], ad_itermax=25, ppe_itermax=100000)
        return dict(case=case, c=c, u=u, v=v, p=p)
    if case["kind"] == "flow":
        return dict(case=case, flow=_flow_input(case, seed))
    return dict(case=case, requests=_requests(case, seed))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _repin(handle, check):
    r = handle.autotune()
    handle.tune(r["kernel"], r["tile_y"], r["sweeps_per_launch"], check)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "compat_ad":
        c = state["c"]
        c.set("u", state["u"])
        c.set("v", state["v"])
        iters = 0
        for _ in range(case["steps"]):
            st = c.ad_step()
            iters += st["ad_iters"]
        return dict(u=c.get("u"), v=c.get("v"), iters=iters, res=st["ad_res"])
    if kind == "compat_ppe":
        c = state["c"]
        c.set("p", state["p"])
        st = c.ppe_solve()
        return dict(p=c.get("p"), sweeps=st["ppe_sweeps"])
    if kind == "flow":
        f = state["flow"]
        with iff.Case(f["xf"], f["yf"], precision=PRECISION[case["precision"]], dt=f["dt"], re=f["re"],
                      bodies=f["bodies"], ad_itermax=25, ad_tol=1e-6, ppe_solver=SOLVER[case["solver"]],
                      ppe_omega=case["omega"], ppe_itermax=400000, ppe_tol=case["tol"], check_every=case["check"]) as c:
            if case["tuned"]:
                first = c.step(1)
                _repin(c, case["check"])
                st = c.step(case["steps"] - 1)
                sweeps = first["total_ppe_sweeps"] + st["total_ppe_sweeps"]
            else:
                st = c.step(case["steps"])
                sweeps = st["total_ppe_sweeps"]
            return dict(u=c.get("u"), v=c.get("v"), p=c.get("p"), sweeps=sweeps, ad_iters=st["ad_iters"])
    b = iff.Batch(PRECISION[case["precision"]])
    try:
        b.tune(4, 64, 8, case["check"])
        slots = [b.add(r["xf"], r["yf"], case["steps"], dt=r["dt"], re=r["re"], bodies=r["bodies"], ppe_tol=case["tol"],
                       ad_itermax=25, check_every=case["check"]) for r in state["requests"]]
        b.step(1)
        _repin(b, case["check"])
        b.step(case["steps"] - 1)
        out = dict(sweeps=np.array([b.state(s)[2]["total_ppe_sweeps"] for s in slots]))
        for k, s in enumerate(slots):
            for name in ("u", "v", "p"):
                out["%s%02d" % (name, k)] = b.get(s, name)
        return out
    finally:
        b.close()


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _sweeps(n, steps):
    """Poisson sweeps of a job's first steps on an n-cell-wide grid: counted,
    3 n to 9 n a step, about 5 n at the middle of the range."""
    return 5.0 * n * steps


def _flow_work(nx, ny, steps, solver="rbsor"):
    cells = float(nx) * ny
    b = cells * 24.0   # u, v, p handed over; the grid and the bodies are small
    per = 9.0 if solver == "rbsor" else 18.0
    sweeps = _sweeps(max(nx, ny), steps) * (1.0 if solver == "rbsor" else 0.6)
    return b, cells * (sweeps * per + steps * (60.0 + 25.0 * 24.0))


def work(case):
    if case["kind"] == "compat_ad":
        cells = (case["nx"] + 2.0) * (case["ny"] + 2.0)
        return {"bytes": cells * 8.0 * 4.0, "flops": cells * case["steps"] * (60.0 + 5.0 * 24.0)}
    if case["kind"] == "compat_ppe":
        cells = (case["nx"] + 2.0) * (case["ny"] + 2.0)
        return {"bytes": cells * 8.0 * 2.0, "flops": cells * 18.0 * 5.9 * max(case["nx"], case["ny"]) ** 2}
    if case["kind"] == "flow":
        ny = case["n"] // 2 if case["grid"] == "stretched" else case["n"]
        b, f = _flow_work(case["n"], ny, case["steps"], case["solver"])
        return {"bytes": b, "flops": f}
    b = f = 0.0
    for k in range(case["count"]):
        n = case["lo"] * (case["hi"] / case["lo"]) ** ((k + 0.5) / case["count"])
        x, y = _flow_work(n, n, case["steps"])
        b, f = b + x, f + y
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same in plain torch / numpy, 64 bits
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _axis(xf):
    """Widths of the cells, ghost copies included, as a float64 tensor."""
    d = np.diff(xf)
    return torch.tensor(np.concatenate((d[:1], d, d[-1:])), dtype=torch.float64, device=_device())


def _edges(q, bc):
    """Dirichlet ghosts q_g = 2 bc - q_in on the four sides, corners kept."""
    q[1:-1, 0] = 2.0 * bc - q[1:-1, 1]
    q[1:-1, -1] = 2.0 * bc - q[1:-1, -2]
    q[0, 1:-1] = 2.0 * bc - q[1, 1:-1]
    q[-1, 1:-1] = 2.0 * bc - q[-2, 1:-1]


class _Stencil:
    """Metric of a grid, and the predictor's stencils on (ny, nx) fields."""

    def __init__(self, xf, yf, dt, re):
        self.dx, self.dy, self.dt = _axis(xf), _axis(yf), dt
        d, e = self.dx, self.dy
        self.cxp, self.cxm = (2.0 / (d[1:-1] * (d[1:-1] + d[k]))[None, :] for k in (slice(2, None), slice(0, -2)))
        self.cyp, self.cym = (2.0 / (e[1:-1] * (e[1:-1] + e[k]))[:, None] for k in (slice(2, None), slice(0, -2)))
        self.nu = dt / re

    def east(self, q):
        """Face values of the interior rows' vertical faces (ny-2, nx-1)."""
        d = self.dx
        return (q[1:-1, 1:] * d[None, :-1] + q[1:-1, :-1] * d[None, 1:]) / (d[:-1] + d[1:])[None, :]

    def north(self, q):
        e = self.dy
        return (q[1:, 1:-1] * e[:-1, None] + q[:-1, 1:-1] * e[1:, None]) / (e[:-1] + e[1:])[:, None]

    def source(self, q, uf, vf):
        fx, fy = self.east(q) * uf, self.north(q) * vf
        return (q[1:-1, 1:-1] - 0.5 * self.dt * (fx[:, 1:] - fx[:, :-1]) / self.dx[None, 1:-1]
                - 0.5 * self.dt * (fy[1:, :] - fy[:-1, :]) / self.dy[1:-1, None])

    def jacobi(self, q, s):
        t = s + self.nu * (self.cxp * q[1:-1, 2:] + self.cxm * q[1:-1, :-2] + self.cyp * q[2:, 1:-1]
                           + self.cym * q[:-2, 1:-1])
        return t / (1.0 + self.nu * (self.cxp + self.cxm + self.cyp + self.cym))


def _exact_compat_ad(case, seed):
    """The reference's ADsolver as coded: stale north-face velocities (its vf
    loop is empty unless nx > ny, so they stay zero there)."""
    nx, ny = case["nx"] + 2, case["ny"] + 2
    if nx > ny:
        return None
    xf, yf, u, v, _ = _compat_fields(case, seed)
    s = _Stencil(xf, yf, case["dt"], case["re"])
    q = [torch.tensor(f.reshape(ny, nx), dtype=torch.float64, device=_device()) for f in (u, v)]
    bc = (1.0, 0.0)
    vf = torch.zeros((ny - 1, nx - 2), dtype=torch.float64, device=_device())

    def bound(f, b):
        old = f[1, 0].clone()
        _edges(f, b)
        f[0, 0] = 2.0 * b - old
        f[-1, 0] = 2.0 * b - f[-2, 0]
        f[-1, -1] = 2.0 * b - f[-2, -1]
        f[0, -1] = 2.0 * b - f[0, -2]

    iters = 0
    for _ in range(case["steps"]):
        uf = s.east(q[0])
        for f, b in zip(q, bc):
            bound(f, b)
        src = [s.source(f, uf, vf) for f in q]
        spare = [torch.zeros_like(f) for f in q]
        res, it = 1.0, 0
        while res > 1e-6 and it < 25:
            for f, b in zip(q, bc):
                bound(f, b)
            for f, g, r in zip(q, spare, src):
                g[1:-1, 1:-1] = s.jacobi(f, r)
            for f, b in zip(q, bc):
                bound(f, b)
            res = float(sum((g - f)[1:-1, 1:-1].abs().sum() for f, g in zip(q, spare)))
            q, spare = spare, q
            it += 1
        iters += it
    return dict(u=q[0].reshape(-1), v=q[1].reshape(-1), iters=None, res=None)


def _exact_compat_ppe(case, seed):
    """Point Jacobi until the signed sum of A p falls to 1e-6."""
    nx, ny = case["nx"] + 2, case["ny"] + 2
    if max(nx, ny) > 64:
        return None
    xf, yf, _, _, p = _compat_fields(case, seed)
    d, e = (np.concatenate((w[:1], w, w[-1:])) for w in (np.diff(xf), np.diff(yf)))
    cxp, cxm = (2.0 / (d[1:-1] * (d[1:-1] + d[k])) for k in (slice(2, None), slice(0, -2)))
    cyp, cym = (2.0 / (e[1:-1] * (e[1:-1] + e[k]))[:, None] for k in (slice(2, None), slice(0, -2)))
    ap = (cxp + cxm)[None, :] + (cyp + cym)
    p = p.reshape(ny, nx).copy()
    p[:, 0] = p[0, :] = 100.0
    for _ in range(100000):
        p[1:-1, 1:-1] = (p[1:-1, 2:] * cxp + p[1:-1, :-2] * cxm + p[2:, 1:-1] * cyp + p[:-2, 1:-1] * cym) / ap
        r = (p[1:-1, 2:] * cxp + p[1:-1, :-2] * cxm + p[2:, 1:-1] * cyp + p[:-2, 1:-1] * cym) - ap * p[1:-1, 1:-1]
        if r.sum() <= 1e-6:
            break
    p[:, 0] = p[0, :] = 100.0
    return dict(p=p.reshape(-1), sweeps=None)


def _circle_ghosts(xc, yc, fluid, body):
    """Ghost cells of a circle (solid cells next to the fluid) and the weights
    of their image points' bilinear stencils: (index, nodes, wd, wn)."""
    ny, nx = fluid.shape
    near = np.zeros_like(fluid)
    near[1:-1, 1:-1] = fluid[1:-1, 2:] | fluid[1:-1, :-2] | fluid[2:, 1:-1] | fluid[:-2, 1:-1]
    j, i = np.nonzero(near & ~fluid)
    gx, gy = xc[i], yc[j]
    ex, ey = gx - body["xc"], gy - body["yc"]
    dist = np.hypot(ex, ey)
    ipx = 2.0 * (body["xc"] + body["r"] * ex / dist) - gx
    ipy = 2.0 * (body["yc"] + body["r"] * ey / dist) - gy
    i0, j0 = np.searchsorted(xc, ipx, side="right") - 1, np.searchsorted(yc, ipy, side="right") - 1
    fx, fy = (ipx - xc[i0]) / (xc[i0 + 1] - xc[i0]), (ipy - yc[j0]) / (yc[j0 + 1] - yc[j0])
    me = j * nx + i
    nodes = np.stack([j0 * nx + i0, j0 * nx + i0 + 1, (j0 + 1) * nx + i0, (j0 + 1) * nx + i0 + 1])
    w = np.stack([(1 - fx) * (1 - fy), fx * (1 - fy), (1 - fx) * fy, fx * fy])
    own = nodes == me
    fl = fluid.reshape(-1)[nodes] & ~own
    wself, wfluid = (w * own).sum(0), (w * fl).sum(0)
    wd = np.where(fl, -w / (1.0 + wself), 0.0)
    wn = np.where(fl, w / np.where(wfluid > 0, wfluid, 1.0), 0.0)
    dev = _device()
    return [torch.tensor(a, device=dev) for a in (me, nodes, wd, wn)]


def _exact_flow(case, seed):
    """The fractional step around one resting circle in 64 bits: explicit
    convection, Jacobi for the implicit viscous part, red-black SOR for the
    pressure with a check of dt |b - A p| every few sweeps, projection."""
    if (case["precision"] != "fp64" or case["solver"] != "rbsor" or case["body"] != "circle"
            or case["n"] > 300 or case["tuned"]):
        return None
    dev = _device()
    if dev.type == "cpu" and case["n"] > 64:
        return None
    f = _flow_input(case, seed)
    xf, yf, dt, body = f["xf"], f["yf"], f["dt"], f["bodies"][0]
    s = _Stencil(xf, yf, dt, f["re"])
    xc = np.concatenate(([-0.5 * (xf[0] + xf[1])], 0.5 * (xf[:-1] + xf[1:]), [0.0]))
    xc[-1] = 2.0 * xf[-1] - xc[-2]
    yc = np.concatenate(([-0.5 * (yf[0] + yf[1])], 0.5 * (yf[:-1] + yf[1:]), [0.0]))
    yc[-1] = 2.0 * yf[-1] - yc[-2]
    nx, ny = len(xc), len(yc)
    ex, ey = xc[None, :] - body["xc"], yc[:, None] - body["yc"]
    fluid = ~(ex * ex + ey * ey <= body["r"] * body["r"])
    gi, gn, gwd, gwn = _circle_ghosts(xc, yc, fluid, body)
    fl = torch.tensor(fluid, device=dev)
    inner = fl[1:-1, 1:-1].to(torch.float64)

    def t(*shape):
        return torch.zeros(shape, dtype=torch.float64, device=dev)

    # open faces join two interior fluid cells
    oe, on = t(ny - 2, nx - 1), t(ny - 1, nx - 2)
    oe[:, 1:-1] = (fl[1:-1, 1:-2] & fl[1:-1, 2:-1]).to(torch.float64)
    on[1:-1, :] = (fl[1:-2, 1:-1] & fl[2:-1, 1:-1]).to(torch.float64)

    def ghost_vel(q):
        q = q.reshape(-1)
        q[gi] = (gwd * q[gn]).sum(0)

    def faces(u, v):
        uf, vf = s.east(u) * oe, s.north(v) * on
        uf[:, 0] = uf[:, -1] = 1.0
        return uf, vf

    u, v, p = t(ny, nx), t(ny, nx), t(ny, nx)
    u[fl] = 1.0
    _edges(u, 1.0)
    _edges(v, 0.0)
    ghost_vel(u)
    ghost_vel(v)
    uf, vf = faces(u, v)

    ae, aw, an, as_ = s.cxp * oe[:, 1:], s.cxm * oe[:, :-1], s.cyp * on[1:, :], s.cym * on[:-1, :]
    sa = (ae + aw) + (an + as_)
    om = 2.0 / (1.0 + math.sin(math.pi / max(nx - 2, ny - 2)))
    act = (sa > 0) & fl[1:-1, 1:-1]
    w = torch.where(act, om / torch.where(sa > 0, sa, torch.ones_like(sa)), torch.zeros_like(sa))
    jj, ii = torch.meshgrid(torch.arange(1, ny - 1, device=dev), torch.arange(1, nx - 1, device=dev), indexing="ij")
    colour = [((ii + jj) % 2 == k) & act for k in (0, 1)]
    wc = [torch.where(m, w, torch.zeros_like(w)) for m in colour]
    keep = [torch.where(m, torch.full_like(w, 1.0 - om), torch.ones_like(w)) for m in colour]

    def apply(p):
        return (ae * p[1:-1, 2:] + aw * p[1:-1, :-2]) + (an * p[2:, 1:-1] + as_ * p[:-2, 1:-1])

    sweeps = iters = 0
    for _ in range(case["steps"]):
        src = s.source(u, uf, vf), s.source(v, uf, vf)
        res, iters = 1.0, 0
        while res > 1e-6 and iters < 25:
            new = []
            for q, r, b in ((u, src[0], 1.0), (v, src[1], 0.0)):
                g = q.clone()
                g[1:-1, 1:-1] = s.jacobi(q, r) * inner
                _edges(g, b)
                ghost_vel(g)
                new.append(g)
            res = float(((new[0] - u)[1:-1, 1:-1].abs() * inner).sum() + ((new[1] - v)[1:-1, 1:-1].abs() * inner).sum())
            u, v = new
            iters += 1
        uf, vf = faces(u, v)
        rhs = ((uf[:, 1:] - uf[:, :-1]) / s.dx[None, 1:-1] + (vf[1:, :] - vf[:-1, :]) / s.dy[1:-1, None]) / dt * inner
        zero = torch.zeros_like(rhs)
        for _ in range(100000):
            r = torch.where(act, rhs - (apply(p) - sa * p[1:-1, 1:-1]), zero)
            if not dt * float(r.abs().max()) > case["tol"]:
                break
            for _ in range(case["check"]):
                for k in (0, 1):
                    pin = p[1:-1, 1:-1]
                    pin.copy_(keep[k] * pin + wc[k] * (apply(p) - rhs))
            sweeps += case["check"]
        p[1:-1, 0], p[1:-1, -1], p[0, 1:-1], p[-1, 1:-1] = p[1:-1, 1], p[1:-1, -2], p[1, 1:-1], p[-2, 1:-1]
        p.reshape(-1)[gi] = (gwn * p.reshape(-1)[gn]).sum(0)
        d, e = s.dx, s.dy
        uf = uf - dt * oe * (p[1:-1, 1:] - p[1:-1, :-1]) * (2.0 / (d[1:] + d[:-1]))[None, :]
        vf = vf - dt * on * (p[1:, 1:-1] - p[:-1, 1:-1]) * (2.0 / (e[1:] + e[:-1]))[:, None]
        px, py = s.east(p), s.north(p)
        u[1:-1, 1:-1] = inner * (u[1:-1, 1:-1] - dt * (px[:, 1:] - px[:, :-1]) / d[None, 1:-1])
        v[1:-1, 1:-1] = inner * (v[1:-1, 1:-1] - dt * (py[1:, :] - py[:-1, :]) / e[1:-1, None])
        for q, b in ((u, 1.0), (v, 0.0)):
            _edges(q, b)
            ghost_vel(q)
    return dict(u=u.reshape(-1), v=v.reshape(-1), p=p.reshape(-1), sweeps=None, ad_iters=None)


def exact(case, seed):
    if case["kind"] == "compat_ad":
        return _exact_compat_ad(case, seed)
    if case["kind"] == "compat_ppe":
        return _exact_compat_ppe(case, seed)
    if case["kind"] == "flow":
        return _exact_flow(case, seed)
    return None

"""What a user of this framework has it compute, as cases to time and compare.

A case is one of four kinds of work:

* ``run``       ``Model.run`` from a host state to a host state, the
                reference's own way of running an experiment: CFL steps, a
                host check after every solve, small grids;
* ``steps``     a resident model advanced by ``device_steps`` (production
                runs: nothing leaves the device between the steps);
* ``ensemble``  many qgrsw basins of uneven sizes advanced together;
* ``gradient``  a final-time misfit and its gradient with respect to the
                initial vorticity (``EulerGradient`` under autograd).

Every pass starts from the same initial state, so that it can be repeated.
``exact`` computes a pass in float64 with plain torch: the discretisation
written out again, the elliptic solves by dense eigenvector transforms of
the rectangle (and conjugate gradients preconditioned with them on a mask).
"""
import math

import numpy as np
import torch

H = 3  # halo cells


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def _case(name, kind, model, nx, ny, domain="closed", land="none", precision="fp64",
          steps=8, members=""):
    c = dict(kind=kind, model=model, nx=nx, ny=ny, domain=domain, land=land,
             precision=precision, steps=steps, members=members)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the default Param (40^2, closed, euler) with the dipole of the
        # reference's own example and test, run to t = 10: the smallest grid,
        # bound by launches and host checks
        _case("dipole_run_40", "run", "euler", 40, 40, steps=22),
        # the closed 256^2 vortex (Gaussian vortex plus noise), as an
        # experiment script runs it: Model.run with CFL steps
        _case("vortex_run_256", "run", "eulerpsi", 256, 256, steps=24),
        # free turbulence on the torus, the benchmark's size, both precisions
        _case("turbulence_1024_fp64", "steps", "eulerpsi", 1024, 1024, "periodic", steps=16),
        _case("turbulence_1024_fp32", "steps", "eulerpsi", 1024, 1024, "periodic",
              precision="fp32", steps=16),
        # the same flow at the largest grid: production resolution
        _case("turbulence_4096_fp64", "steps", "eulerpsi", 4096, 4096, "periodic", steps=4),
        # a channel of sizes picked by a domain's proportions and not by
        # powers of two
        _case("channel_800x304", "steps", "eulerpsi", 800, 304, "channel", steps=8),
        # a wind-driven-gyre-like basin with a coastline on the beta plane
        _case("gyre_basin_512", "steps", "qg", 512, 512, land="basin", steps=8),
        # momentum-pressure Euler around islands: the masked pressure
        # projection of the reference's default model
        _case("islands_euler_192x160", "steps", "euler", 192, 160, land="islands", steps=4),
        # the shallow-water island channel of the benchmark, FP32
        _case("channel_rsw_2048x1024", "steps", "rsw", 2048, 1024, "channel", "islands",
              "fp32", steps=16),
        # a smaller shallow-water domain of odd sizes in FP64
        _case("rsw_501x333", "steps", "rsw", 501, 333, "closed", "islands", steps=16),
        # an ensemble of basins of uneven sizes
        _case("ensemble_qgrsw", "ensemble", "qgrsw", 512, 512, land="basin",
              precision="fp32", steps=8,
              members="512,512,512,256,256,256,256,128,128,128,128,128"),
        # gradient of the final-time misfit, 60 steps with checkpoints
        _case("gradient_512", "gradient", "eulerpsi", 512, 512, "periodic",
              precision="fp32", steps=60),
    ]


def _side(rng, lo, hi):
    """A grid side, spread over its logarithm: any number, or (as users
    often choose) a power of two or a multiple of 20."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    style = rng.random()
    if style < 0.25:
        return int(min(hi, max(lo, 2 ** round(math.log2(n)))))
    if style < 0.45:
        return int(min(hi, max(lo, 20 * round(n / 20))))
    return int(round(n))


def _even_side(rng, lo, hi):
    """A grid side for a model with an elliptic solve: an odd factor up to
    25 times a power of two (a multigrid hierarchy needs a small coarsest
    level), a power of two in a third of them."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    odd = 1 if rng.random() < 1 / 3 else rng.choice([3, 5, 7, 9, 11, 13, 15, 17, 19, 21, 23, 25])
    k = max(2, round(math.log2(n / odd)))
    while odd * 2 ** k > hi:
        k -= 1
    while odd * 2 ** k < lo:
        k += 1
    return odd * 2 ** k


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["run"] * 2 + ["steps"] * 7 + ["ensemble", "gradient"])
    if kind == "ensemble":
        sizes = [_even_side(rng, 64, 512) for _ in range(rng.randint(1, 4))]
        sizes = sorted((n for n in sizes for _ in range(rng.randint(1, 4))), reverse=True)
        return _case("", kind, "qgrsw", sizes[0], sizes[0], land="basin", precision="fp32",
                     steps=2 * rng.randint(2, 4), members=",".join(map(str, sizes)))
    if kind == "gradient":
        n = 2 ** rng.randint(6, 9)
        return _case("", kind, "eulerpsi", n, n * rng.choice([1, 1, 2]), "periodic",
                     precision=rng.choice(["fp64", "fp32", "fp32"]), steps=rng.randint(10, 60))
    model = rng.choice(["euler", "eulerpsi", "advection", "qg", "rsw"]) if kind == "run" else \
        rng.choice(["eulerpsi"] * 4 + ["qg", "advection", "euler", "rsw", "rsw"])
    side = _side if model in ("advection", "rsw") else _even_side
    if kind == "run":
        nx = side(rng, 40, 200 if model == "euler" else 320)
        ny = nx if rng.random() < 0.5 else side(rng, 36, nx)
        land = "islands" if rng.random() < 0.25 and model != "advection" else "none"
        return _case("", kind, model, nx, ny, "closed", land, "fp64", rng.randint(8, 24))
    lo, hi = (48, 320) if model == "euler" else (64, 1600)
    nx = side(rng, lo, hi)
    ny = nx if rng.random() < 0.4 else side(rng, max(lo, nx / 2), min(hi, nx * 2))
    domain = rng.choice(["closed", "channel"] + (["periodic"] * 2 if model == "eulerpsi" else []))
    land = "none" if domain == "periodic" or model == "advection" else \
        rng.choice(["none", "none", "islands", "basin" if domain == "closed" else "islands"])
    precision = rng.choice(["fp64", "fp32"]) if model in ("eulerpsi", "rsw", "advection") \
        else "fp64"
    return _case("", kind, model, nx, ny, domain, land, precision, 4 * rng.randint(1, 3))


# --------------------------------------------------------------------------
# geometry and initial fields (host, float64)
# --------------------------------------------------------------------------
def _lengths(case):
    """Lx, Ly of square cells, the longer side 1."""
    n = max(case["nx"], case["ny"])
    return case["nx"] / n, case["ny"] / n


def _fill(a, xper, yper):
    if xper:
        a[..., :H] = a[..., -2 * H:-H]
        a[..., -H:] = a[..., H:2 * H]
    if yper:
        a[..., :H, :] = a[..., -2 * H:-H, :]
        a[..., -H:, :] = a[..., H:2 * H, :]
    return a


def _periods(case):
    return case["domain"] in ("channel", "periodic"), case["domain"] == "periodic"


def _coords(nx, ny, at):
    """Coordinates on the padded grid in units of the longer side."""
    n = max(nx, ny)
    s = 0.5 if at == "c" else 0.0
    return np.meshgrid((np.arange(nx + 2 * H) - H + s) / n, (np.arange(ny + 2 * H) - H + s) / n)


def _mask(case, nx, ny):
    """The cell mask of the case's coastline (the same for every seed)."""
    xper, yper = _periods(case)
    m = np.zeros((ny + 2 * H, nx + 2 * H), dtype=np.int8)
    m[slice(None) if yper else slice(H, -H), slice(None) if xper else slice(H, -H)] = 1
    x, y = _coords(nx, ny, "c")
    rng = np.random.default_rng([nx, ny])
    lx, ly = nx / max(nx, ny), ny / max(nx, ny)
    if case["land"] == "basin":  # one bay-and-cape coastline around the middle
        th = np.arctan2((y - ly / 2) / ly, (x - lx / 2) / lx)
        r = np.hypot((y - ly / 2) / ly, (x - lx / 2) / lx)
        coast = 0.4 + sum(0.02 * rng.uniform(-1, 1) * np.cos(k * th + rng.uniform(0, 6.28))
                          for k in range(2, 7))
        m[r > coast] = 0
    elif case["land"] == "islands":
        small = min(lx, ly)
        for _ in range(6):
            r = small * rng.uniform(0.02, 0.07)
            cx, cy = rng.uniform(0, lx), rng.uniform(0.15 * ly, 0.85 * ly)
            ddx = np.abs(x - cx)
            if xper:
                ddx = np.minimum(ddx, lx - ddx)
            m[ddx ** 2 + (y - cy) ** 2 < r * r] = 0
    return _fill(m, xper, yper)


def _smooth(x, y, lx, ly, rng, k0=8.0, kmax=20):
    """Random-phase field with a k^-3 exp(-(k/k0)^2) energy spectrum of the
    vorticity's flow, unit RMS, periodic on the domain."""
    kx, ky = np.arange(kmax + 1), np.arange(kmax + 1)
    k = np.hypot(kx[None, :], ky[:, None])
    k[0, 0] = np.inf
    amp = np.sqrt(k ** -3 * np.exp(-(np.minimum(k, 1e3) / k0) ** 2))
    amp = np.where(np.isfinite(k), amp, 0.0)
    ex, ey = 2 * np.pi * np.outer(kx, x[0] / lx), 2 * np.pi * np.outer(ky, y[:, 0] / ly)
    w = 0.0
    for fy in (np.cos, np.sin):
        for fx in (np.cos, np.sin):
            w = w + fy(ey).T @ (amp * rng.standard_normal(amp.shape)) @ fx(ex)
    return w / np.sqrt(np.mean(w[H:-H, H:-H] ** 2))


def _bumps(x, y, lx, ly, rng, count=6):
    out = np.zeros_like(x)
    for _ in range(count):
        x0, y0 = rng.uniform(0.25, 0.75, 2) * (lx, ly)
        r = rng.uniform(0.03, 0.08) * min(lx, ly)
        out += rng.choice([-1, 1]) * np.exp(-((x - x0) ** 2 + (y - y0) ** 2) / (2 * r * r))
    return out


def _initial(case, nx, ny, seed):
    """The field an experiment script sets, on the padded grid: vorticity
    (euler, at the vertices; eulerpsi), potential vorticity (qg), tracer
    (advection) or thickness (rsw, qgrsw), times the cell area, unmasked."""
    rng = np.random.default_rng([seed, nx, ny])
    lx, ly = nx / max(nx, ny), ny / max(nx, ny)
    area = 1.0 / max(nx, ny) ** 2
    model = case["model"]
    x, y = _coords(nx, ny, "v" if model == "euler" else "c")
    if model == "euler":  # the dipole, its place and axis by seed
        x0, y0 = lx * rng.uniform(0.4, 0.6), ly * rng.uniform(0.4, 0.6)
        a, d, r = rng.uniform(0, 6.28), 0.05, 0.05
        g = [np.exp(-((x - x0 - s * d * np.cos(a)) ** 2 + (y - y0 - s * d * np.sin(a)) ** 2)
                    / (2 * r * r)) for s in (1, -1)]
        f = g[0] - g[1]
    elif model in ("rsw", "qgrsw"):
        f = 1.0 + 0.05 * _bumps(x, y, lx, ly, rng)
    elif case["kind"] == "run" and model == "eulerpsi":
        f = np.exp(-((x - lx / 2) ** 2 + (y - ly / 2) ** 2) / (2 * 0.1 ** 2)) \
            + 1e-3 * rng.uniform(-1, 1, x.shape)
    else:
        f = _smooth(x, y, lx, ly, rng)
    return _fill(f * area, *_periods(case))


def _planetary(case, nx, ny):
    """beta-plane vorticity at the vertices times the area (qg)."""
    _, y = _coords(nx, ny, "v")
    return 2.0 * (y - 0.5) / max(nx, ny) ** 2


def _rotation(case, nx, ny):
    """Streamfunction of the advection model's fixed flow, at the vertices
    (0 on the walls)."""
    x, y = _coords(nx, ny, "v")
    lx, ly = _lengths(case)
    s = np.sin(np.pi * y / ly) ** 2
    if not _periods(case)[0]:
        s = s * np.sin(np.pi * x / lx) ** 2
    return s / (2 * np.pi)


F0, GRAV, DEPTH, CFL = 10.0, 1.0, 1.0, 0.9


def _dt(case):
    """The fixed step of a resident run (0: the CFL step)."""
    if case["kind"] == "run" or case["model"] == "rsw":
        return 0.0
    n = max([case["nx"], case["ny"]])
    if case["model"] == "qgrsw":
        return 0.02  # f0 dt = 0.2: the flow is slow
    if case["model"] == "advection":
        return 0.4 / n
    return 0.9 / n


# --------------------------------------------------------------------------
# the framework's side
# --------------------------------------------------------------------------
def _param(case, nx, ny):
    import fluids2d_amd.param as fp
    fp.QUIET = True
    from fluids2d_amd import Param
    p = Param()
    p.model, p.nx, p.ny = case["model"], nx, ny
    n = max(nx, ny)
    p.Lx, p.Ly = nx / n, ny / n
    p.xperiodic, p.yperiodic = _periods(case)
    p.f0, p.g, p.H, p.cfl = F0, GRAV, DEPTH, CFL
    p.beta = 1.0 if case["model"] == "qg" else 0.0
    p.dt = _dt(case)
    p.tend, p.maxite, p.nprint = 1e30, 10 ** 9, 10 ** 9
    p.precision = case["precision"]
    return p


def _model(case, nx, ny, seed):
    """A Model with its coastline and initial state, its diagnostics done."""
    from fluids2d_amd import Model
    from fluids2d_amd.rsw import qg_projection
    from fluids2d_amd.tools import set_uv_from_omega
    m = Model(_param(case, nx, ny))
    mesh, s, kind = m.mesh, m.state, case["model"]
    if case["land"] != "none":
        mesh.msk[...] = _mask(case, nx, ny)
        mesh.finalize()
    f = _initial(case, nx, ny, seed)
    if kind == "euler":
        set_uv_from_omega(m, f * mesh.mskv, s.u)
    elif kind == "advection":
        s.q[...] = f * mesh.msk
        psi = _rotation(case, nx, ny) * mesh.mskv
        s.U.x[:-1] = -np.diff(psi, axis=0) * mesh.mskx[:-1] / mesh.dy ** 2
        s.U.y[:, :-1] = np.diff(psi, axis=1) * mesh.msky[:, :-1] / mesh.dx ** 2
        mesh.fill(s.U)
    elif kind in ("rsw", "qgrsw"):
        s.h[...] = f * mesh.msk
    else:
        getattr(s, "pv" if kind == "qg" else "omega")[...] = f * mesh.msk
    if kind == "qg":
        mesh.f = _planetary(case, nx, ny)
    if kind == "qgrsw":
        qg_projection(m)
    else:
        m.integrator.diag(s)
    return m


# the fields whose values the next step depends on, per model (a diagnostic
# field that starts an iterative solve among them)
STATE = {"euler": ("u", "U", "omega", "ke", "p"), "eulerpsi": ("omega", "U", "psi"),
         "qg": ("pv", "U", "psi"), "advection": ("q", "U"),
         "rsw": ("u", "h", "U", "omega", "ke", "p"), "qgrsw": ("u", "h", "U", "omega", "psi")}
# the fields a pass returns
RESULT = {"euler": ("u", "omega"), "eulerpsi": ("omega", "psi"), "qg": ("pv", "psi"),
          "advection": ("q",), "rsw": ("u", "h"), "qgrsw": ("u", "h")}


def _arrays(state, names):
    out = []
    for n in names:
        v = getattr(state, n)
        out += [v.x, v.y] if hasattr(v, "x") else [v]
    return out


class _Resident:
    """A model on the device and a copy of its initial device state."""

    def __init__(self, model):
        self.model = model
        self.names = STATE[model.param.model]
        model.integrator.begin(model.state)
        self.start = [a.clone() for a in _arrays(model.integrator.dstate, self.names)]

    def now(self):
        return _arrays(self.model.integrator.dstate, self.names)

    def rewind(self):
        torch._foreach_copy_(self.now(), self.start)

    def result(self):
        return _arrays(self.model.integrator.dstate, RESULT[self.model.param.model])


def prepare(case, seed):
    nx, ny, kind = case["nx"], case["ny"], case["kind"]
    if kind == "run":
        m = _model(case, nx, ny, seed)
        m.param.maxite = case["steps"]
        every = STATE[case["model"]]
        return {"kind": kind, "model": m, "names": every,
                "start": [a.copy() for a in _arrays(m.state, every)]}
    if kind == "steps":
        r = _Resident(_model(case, nx, ny, seed))
        if getattr(r.model.integrator.model, "capturable", True):
            r.model.integrator.prepare_graph()
        r.rewind()
        return {"kind": kind, "resident": r, "steps": case["steps"]}
    if kind == "ensemble":
        from fluids2d_amd.ensemble import Ensemble
        sizes = [int(n) for n in case["members"].split(",")]
        members = [_Resident(_model(case, n, n, seed + 101 * k)) for k, n in enumerate(sizes)]
        ens = Ensemble([r.model for r in members])
        ens.steps(4)
        return {"kind": kind, "members": members, "ensemble": ens, "steps": case["steps"],
                "start": [a for r in members for a in r.start]}
    from fluids2d_amd.adjoint import EulerAdjoint
    p = _param(case, nx, ny)
    runner = EulerAdjoint(p, _dt(case), case["steps"], checkpoint=20)
    w0, goal = (torch.from_numpy(_initial(case, nx, ny, s)).to(runner.mesh.device, runner.dtype)
                for s in (seed, seed + 7919))
    return {"kind": kind, "runner": runner, "omega": w0.requires_grad_(True),
            "goal": 0.5 * (w0.detach() + goal)}


def run(state):
    kind = state["kind"]
    if kind == "run":
        from fluids2d_amd.timeline import Time
        m = state["model"]
        for a, b in zip(_arrays(m.state, state["names"]), state["start"]):
            a[...] = b
        m.time = Time(m.param)
        m.run()
        return {"fields": _arrays(m.state, RESULT[m.param.model]), "ite": m.time.ite}
    if kind == "steps":
        r = state["resident"]
        r.rewind()
        r.model.integrator.device_steps(state["steps"])
        return {"fields": r.result()}
    if kind == "ensemble":
        torch._foreach_copy_([a for r in state["members"] for a in r.now()], state["start"])
        state["ensemble"].steps(state["steps"])
        return {"fields": [a for r in state["members"] for a in r.result()]}
    from fluids2d_amd.adjoint import EulerGradient
    w0 = state["omega"]
    w0.grad = None
    w = EulerGradient.apply(w0, state["runner"])
    _misfit(w, state["goal"]).backward()
    return {"omega": w.detach(), "gradient": w0.grad}


def _misfit(w, goal):
    """Half the squared distance of the interiors, in units of the goal's
    mean square."""
    d = (w - goal)[H:-H, H:-H]
    return 0.5 * (d * d).sum() / (goal[H:-H, H:-H] ** 2).mean()


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    """Per RK stage the prognostic fields are read once and written once;
    the reconstructions take about 70 operations a face (two faces a cell
    and field; the momentum models evaluate six), the solve those of a fast
    transform.  A gradient costs about three such runs."""
    b = 8 if case["precision"] == "fp64" else 4
    grids = [(case["nx"], case["ny"])]
    if case["kind"] == "ensemble":
        grids = [(int(n), int(n)) for n in case["members"].split(",")]
    fields = {"euler": 2, "rsw": 3, "qgrsw": 3}.get(case["model"], 1)
    faces = {"euler": 4, "rsw": 6, "qgrsw": 4}.get(case["model"], 2)
    stages = 3 * case["steps"] * (3 if case["kind"] == "gradient" else 1)
    by = fl = 0.0
    for nx, ny in grids:
        solve = 0 if case["model"] in ("rsw", "advection") else 10 * math.log2(nx * ny)
        by += stages * nx * ny * 2 * b * fields
        fl += stages * nx * ny * (70 * faces + solve)
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """FP64: rounding (1e-13 in the fields) and the solves' 1e-13 relative
    residuals, which the streamfunction of a large grid shows as up to 1e-10.
    FP32: rounding of the fields (1e-7 to 2e-6 off float64); the shallow-water
    velocity starts from rest and sums differences of a thickness near 1, so
    it is 5e-5 to 2e-4 off; the gradient (2e-6 off) crosses kinks of the
    reconstruction's weights."""
    if case["precision"] == "fp64":
        return {"rel": 1e-9, "max": 1e-7}
    if case["model"] == "rsw":
        return {"rel": 8e-4, "max": 5e-2}
    if case["kind"] == "gradient":
        return {"rel": 1e-4, "max": 1e-2}
    return {"rel": 1e-5, "max": 1e-3}


# --------------------------------------------------------------------------
# the same pass in float64 with plain torch
# --------------------------------------------------------------------------
def _basis(n, bc, dev):
    """Orthonormal eigenvectors (columns) and eigenvalues of the second
    difference: sines on n - 1 interior points ("wall"), Fourier modes on n
    points ("ring"), cosines on n cells ("even")."""
    pi = math.pi
    if bc == "wall":
        i = torch.arange(1, n, device=dev, dtype=torch.int64)
        ang = (torch.outer(i, i) % (2 * n)).double() * (pi / n)
        return math.sqrt(2.0 / n) * torch.sin(ang), 2 * torch.cos(i.double() * (pi / n)) - 2
    if bc == "ring":
        i = torch.arange(n, device=dev, dtype=torch.int64)
        k = (i + 1) // 2  # 0, 1, 1, 2, 2, ...
        ang = (torch.outer(i, k) % n).double() * (2 * pi / n)
        q = torch.where(i % 2 == 1, torch.cos(ang), torch.sin(ang))
        q[:, 0] = math.sqrt(0.5)
        if n % 2 == 0:
            q[:, -1] = math.sqrt(0.5) * (1 - 2 * (i % 2)).double()
        return math.sqrt(2.0 / n) * q, 2 * torch.cos(k.double() * (2 * pi / n)) - 2
    i = torch.arange(n, device=dev, dtype=torch.int64)
    ang = (torch.outer(2 * i + 1, i) % (4 * n)).double() * (pi / (2 * n))
    q = math.sqrt(2.0 / n) * torch.cos(ang)
    q[:, 0] *= math.sqrt(0.5)
    return q, 2 * torch.cos(i.double() * (pi / n)) - 2


class _Elliptic:
    """The 5-point operator on the vertices (Dirichlet at the coast) or the
    cells (no flux through the coast), solved by eigenvectors of the
    rectangle, with conjugate gradients around them on a mask."""

    def __init__(self, d, at, mass=0.0):
        self.d, self.at = d, at
        msk = d.mskv if at == "v" else d.msk
        u = msk[H:-H, H:-H].double()
        ny, nx = u.shape
        self.off_x = int(at == "v" and not d.xper)
        self.off_y = int(at == "v" and not d.yper)
        self.u = u
        cx, cy = d.dy / d.dx, d.dx / d.dy
        other = "wall" if at == "v" else "even"
        self.qx, lx = _basis(nx, "ring" if d.xper else other, d.dev)
        self.qy, ly = _basis(ny, "ring" if d.yper else other, d.dev)
        lam = cx * lx[None, :] + cy * ly[:, None] - mass
        self.zero = bool(lam.abs().max() > 0 and lam.abs().min() < 1e-12 * lam.abs().max())
        inv = 1 / torch.where(lam.abs() < 1e-12 * lam.abs().max(), lam.abs().max(), lam)
        dead = lam.abs() < 1e-12 * lam.abs().max()
        whole = u[self.off_y:, self.off_x:]
        self.full = bool((whole == 1).all())
        self.singular = self.zero and (self.full or at == "c")
        self.inv = torch.where(dead, torch.zeros_like(inv), inv) if self.singular else \
            torch.where(dead, 1 / lam.abs().masked_fill(dead, math.inf).min() * -1, inv)
        # face weights: both sides unknown; no wrap through a wall
        self.wx, self.wy = cx * u * torch.roll(u, 1, 1), cy * u * torch.roll(u, 1, 0)
        if not d.xper:
            self.wx[:, 0] = 0
        if not d.yper:
            self.wy[0, :] = 0
        if at == "v":
            self.diag = (2 * cx + 2 * cy + mass) * u
        else:
            self.diag = self.wx + torch.roll(self.wx, -1, 1) + self.wy + torch.roll(self.wy, -1, 0)

    def apply(self, x):
        """-A x (positive)."""
        wx, wy = self.wx, self.wy
        return self.diag * x - (wx * torch.roll(x, 1, 1) + torch.roll(wx * x, -1, 1)
                                + wy * torch.roll(x, 1, 0) + torch.roll(wy * x, -1, 0))

    def direct(self, b):
        out = torch.zeros_like(b)
        c = self.qy.T @ b[self.off_y:, self.off_x:] @ self.qx
        out[self.off_y:, self.off_x:] = self.qy @ (c * self.inv) @ self.qx.T
        return out

    def solve(self, b, first=None):
        """x with A x = b at the unknowns, on a padded array (autograd goes
        through the direct form)."""
        g = b[H:-H, H:-H] * self.u
        if self.singular:
            g = (g - g.sum() / self.u.sum()) * self.u
        if self.full:
            x = self.direct(g)
        else:
            x = self._cg(-g)
        if self.singular:
            x = (x - (x * self.u).sum() / self.u.sum()) * self.u
        return self.d.pad(x)

    def _cg(self, g):
        x = torch.zeros_like(g)
        r, p, rz = g.clone(), None, None
        norm, best = float(g.norm()), math.inf
        for it in range(1000):
            z = -self.direct(r) * self.u
            if self.singular:
                z = (z - (z * self.u).sum() / self.u.sum()) * self.u
            new = (r * z).sum()
            p = z if p is None else z + (new / rz) * p
            rz = new
            q = self.apply(p)
            a = rz / (p * q).sum()
            x, r = x + a * p, r - a * q
            if it % 8 == 7:
                err = float(r.norm())
                if err <= 1e-15 * norm or not err < best * 2:
                    break
                best = min(best, err)
        return x


class _Domain:
    """Masks, stencil orders and operators on padded float64 arrays."""

    def __init__(self, case, nx, ny, dev):
        self.dev, self.case = dev, case
        self.xper, self.yper = _periods(case)
        self.nx, self.ny = nx, ny
        n = max(nx, ny)
        self.dx, self.dy = nx / n / nx, ny / n / ny
        self.area = self.dx * self.dy
        m = torch.from_numpy(_mask(case, nx, ny)).to(dev).long()
        self.msk = m
        self.s = m.shape[1]  # shift of one row
        zx, zy = torch.zeros_like(m[:, :1]), torch.zeros_like(m[:1])
        west, south = torch.cat([zx, m[:, :-1]], 1), torch.cat([zy, m[:-1]], 0)
        sw = torch.cat([zy, west[:-1]], 0)
        self.mskx, self.msky = m * west, m * south
        self.mskv = m * west * south * sw
        self.slip = ((m + west + south + sw) == 4).double()
        v = (self.slip > 0).long()
        self.oc = self.order(m, 1), self.order(m, self.s)
        self.ov = self.order(v, -1) * self.msky, self.order(v, -self.s) * self.mskx
        self.ok = self.order(self.mskx, -1), self.order(self.msky, -self.s)

    def pad(self, x):
        a = torch.nn.functional.pad(x, (H, H, H, H))
        return self.fill(a)

    def fill(self, a):
        """Halo values of the periodic directions (out of place)."""
        if self.xper:
            a = torch.cat([a[:, -2 * H:-H], a[:, H:-H], a[:, H:2 * H]], 1)
        if self.yper:
            a = torch.cat([a[-2 * H:-H], a[H:-H], a[H:2 * H]], 0)
        return a

    @staticmethod
    def at(a, k):
        """a[i + k] over the flat index."""
        return torch.roll(a.reshape(-1), -k).reshape(a.shape)

    def order(self, m, s):
        """6, 4, 2 or 0: the widest stencil around a face (s > 0: between
        i - s and i; s < 0: between i and i - s) whose points are all wet."""
        flat = m.reshape(-1)

        def wet(k):
            z = torch.zeros_like(flat)
            if k >= 0:
                z[:flat.numel() - k] = flat[k:]
            else:
                z[-k:] = flat[:k]
            return z
        o2 = wet(0) * wet(-s)
        o4 = o2 * wet(-2 * s) * wet(s)
        o6 = o4 * wet(-3 * s) * wet(2 * s)
        return (2 * (o2 + o4 + o6)).reshape(m.shape)

    def face(self, U, q, o, s, first):
        """Upwind WENO reconstruction of q at a face from q[i + (first ...
        first + 5) s]."""
        t = [self.at(q, (first + k) * s) for k in range(6)]
        up = U > 0
        w = [torch.where(up, t[k], t[5 - k]) for k in range(5)]
        f = torch.where(o > 4, _weno5(*w), torch.where(o > 2, _weno3(*w[1:4]), w[2]))
        return torch.where(o > 0, f, torch.zeros_like(f))

    def transport(self, q, U):
        fx = self.face(U[0], q, self.oc[0], 1, -3) * U[0]
        fy = self.face(U[1], q, self.oc[1], self.s, -3) * U[1]
        d = -(self.at(fx, 1) - fx) - (self.at(fy, self.s) - fy)
        return self.fill(d * self.msk)

    def vortex_force(self, U, omega):
        s = self.s
        va = 0.25 * (U[1] + self.at(U[1], s) + self.at(U[1], -1) + self.at(U[1], s - 1))
        vb = 0.25 * (U[0] + self.at(U[0], 1) + self.at(U[0], -s) + self.at(U[0], 1 - s))
        return (self.face(va, omega, self.ov[1], s, -2) * va,
                -self.face(vb, omega, self.ov[0], 1, -2) * vb)

    def coriolis(self, U):
        s, f = self.s, F0 * self.area * 0.25
        cx = U[1] + self.at(U[1], s) + self.at(U[1], -1) + self.at(U[1], s - 1)
        cy = U[0] + self.at(U[0], 1) + self.at(U[0], -s) + self.at(U[0], 1 - s)
        return f * cx, -f * cy

    def grad(self, p):
        return (p - self.at(p, -1)) * self.mskx, (p - self.at(p, -self.s)) * self.msky

    def sharp(self, u):
        return u[0] / self.dx ** 2, u[1] / self.dy ** 2

    def vorticity(self, u):
        w = -(u[0] - self.at(u[0], -self.s)) + (u[1] - self.at(u[1], -1))
        return w * self.slip

    def kinetic(self, u, U):
        s, k = self.s, 0.0
        for c, d in ((0, 1), (1, s)):
            um = 0.5 * (U[c] + self.at(U[c], d))
            k = k + self.face(um, u[c], self.ok[c], d, -2) * um
        return self.fill(k * self.msk * 0.5)

    def to_vertices(self, a):
        s = self.s
        return 0.25 * (a + self.at(a, -1) + self.at(a, -s) + self.at(a, -s - 1)) * self.mskv

    def to_cells(self, v):
        s = self.s
        n = self.mskv + self.at(self.mskv, 1) + self.at(self.mskv, s) + self.at(self.mskv, s + 1)
        t = v + self.at(v, 1) + self.at(v, s) + self.at(v, s + 1)
        return torch.where(self.msk * n > 0, t / n.clamp(min=1), torch.zeros_like(t))

    def perp(self, psi, contra):
        ux = -(self.at(psi, self.s) - psi) * self.mskx
        uy = (self.at(psi, 1) - psi) * self.msky
        if contra:
            ux, uy = ux / self.dy ** 2, uy / self.dx ** 2
        return self.fill(ux), self.fill(uy)


def _weno5(a, b, c, d, e):
    q1 = (2 * a - 7 * b + 11 * c) / 6
    q2 = (-b + 5 * c + 2 * d) / 6
    q3 = (2 * c + 5 * d - e) / 6
    b1 = 13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
    b2 = 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
    b3 = 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
    tau = (b1 - b3).abs()
    w1, w2, w3 = (g * (1 + tau / (x + 1e-16)) for g, x in ((0.1, b1), (0.6, b2), (0.3, b3)))
    return (w1 * q1 + w2 * q2 + w3 * q3) / (w1 + w2 + w3)


def _weno3(a, b, c):
    b1, b2 = (b - a) ** 2, (c - b) ** 2
    tau = (b2 - b1).abs()
    w1, w2 = (1 + tau / (b1 + 1e-14)) / 3, 2 * (1 + tau / (b2 + 1e-14)) / 3
    return (w1 * (1.5 * b - 0.5 * a) + w2 * 0.5 * (b + c)) / (w1 + w2)


class _Flow:
    """One model in float64: prognostic tensors y, tendency and diagnosis."""

    def __init__(self, case, nx, ny, seed, dev):
        self.kind = k = case["model"]
        self.d = d = _Domain(case, nx, ny, dev)
        self.single = case["precision"] == "fp32"
        f = torch.from_numpy(_initial(case, nx, ny, seed)).to(dev)
        mass = d.area * F0 ** 2 / (GRAV * DEPTH) if k in ("qg", "qgrsw") else 0.0
        if k not in ("advection", "rsw"):
            self.ell = _Elliptic(d, "v", mass)
        if k == "euler":
            psi = self.ell.solve(f * d.mskv)
            self.ell = _Elliptic(d, "c")
            self.y = list(d.perp(psi, False))
        elif k == "rsw":
            z = torch.zeros_like(f)
            self.y = [z, z, self._round(f * d.msk)]
        elif k == "qgrsw":
            h = f * d.msk
            w = d.to_vertices((h - DEPTH * d.area) * (-F0 / DEPTH))
            psi = self.ell.solve(w)
            h = (d.to_cells(psi * (F0 * d.area / GRAV)) + DEPTH * d.area) * d.msk
            self.y = [self._round(v) for v in (*d.perp(psi, False), h)]
        else:
            self.y = [self._round(f * d.msk)]
        if k == "advection":
            psi = torch.from_numpy(_rotation(case, nx, ny)).to(dev) * d.mskv
            self.U = tuple(self._round(u) for u in d.perp(psi, True))
        if k == "qg":
            self.f = torch.from_numpy(_planetary(case, nx, ny)).to(dev)
        self.diagnose()

    def _round(self, a):
        """The values a single-precision state holds."""
        return a.float().double() if self.single else a

    def diagnose(self):
        d, k, y = self.d, self.kind, self.y
        if k == "eulerpsi":
            self.psi = self.ell.solve(d.to_vertices(y[0]))
            self.U = d.perp(self.psi, True)
        elif k == "qg":
            self.psi = self.ell.solve(d.to_vertices(y[0]) - self.f)
            self.U = d.perp(self.psi, True)
        elif k in ("euler", "rsw", "qgrsw"):
            if k == "euler":
                U = d.sharp(y[:2])
                div = (d.at(U[0], 1) - U[0] + d.at(U[1], d.s) - U[1]) * d.msk
                g = d.grad(self.ell.solve(div * d.area))
                y[:2] = [d.fill(y[c] - g[c]) for c in (0, 1)]
            self.U = d.sharp(y[:2])
            self.omega = d.fill(d.vorticity(y[:2]))
            if k != "qgrsw":
                self.ke = d.kinetic(y[:2], self.U)

    def tendency(self):
        d, k, y = self.d, self.kind, self.y
        if k in ("eulerpsi", "qg", "advection"):
            return [d.transport(y[0], self.U)]
        a = list(d.vortex_force(self.U, self.omega))
        phi = [self.ke] if k == "euler" else []
        if k != "euler":
            a = [p + q for p, q in zip(a, d.coriolis(self.U))]
        if k == "rsw":
            phi = [self.ke, GRAV / d.area * y[2]]
        for p in phi:
            a = [q - g for q, g in zip(a, d.grad(p))]
        if k == "euler":
            return [d.fill(v) for v in a]
        dh = d.transport(y[2], self.U)
        if k == "qgrsw":
            w = (-(a[0] - d.at(a[0], -d.s)) + (a[1] - d.at(a[1], -1))) * d.slip
            w = w * d.mskv + d.to_vertices(dh * (-F0 / DEPTH))
            psi = self.ell.solve(w)
            a = list(d.perp(psi, False))
            dh = d.to_cells(psi * (F0 * d.area / GRAV)) * d.msk
        return [d.fill(v) for v in (*a, dh)]

    def step(self, dt):
        ds = []
        for coef in ((dt,), (-3 * dt / 4, dt / 4), (-dt / 12, -dt / 12, 2 * dt / 3)):
            ds.append(self.tendency())
            self.y = [v + sum(c * t[i] for c, t in zip(coef, ds)) for i, v in enumerate(self.y)]
            self.diagnose()

    def cfl(self):
        if self.kind == "rsw":
            c = math.sqrt(GRAV * DEPTH)
            return CFL / (c / self.d.dx + c / self.d.dy)
        return CFL / float(self.U[0].abs().max() + self.U[1].abs().max())

    def result(self):
        k, y = self.kind, self.y
        if k in ("eulerpsi", "qg"):
            return [y[0], self.psi]
        return [*y, self.omega] if k == "euler" else list(y)


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    nx, ny, kind = case["nx"], case["ny"], case["kind"]
    if kind == "gradient":
        flow = _Flow(case, nx, ny, seed, dev)
        w0 = flow.y[0].clone().requires_grad_(True)
        goal = flow._round(torch.from_numpy(_initial(case, nx, ny, seed + 7919)).to(dev))
        goal = 0.5 * (w0.detach() + goal)
        flow.y = [flow.d.fill(w0)]
        flow.diagnose()
        for _ in range(case["steps"]):
            flow.step(_dt(case))
        _misfit(flow.y[0], goal).backward()
        return {"omega": flow.y[0].detach(), "gradient": w0.grad}
    if kind == "ensemble":
        sizes = [int(n) for n in case["members"].split(",")]
        flows = [_Flow(case, n, n, seed + 101 * k, dev) for k, n in enumerate(sizes)]
    else:
        flows = [_Flow(case, nx, ny, seed, dev)]
    out = []
    for flow in flows:
        for _ in range(case["steps"]):
            flow.step(_dt(case) or flow.cfl())
        out += flow.result()
    got = {"fields": out}
    if kind == "run":
        got["ite"] = case["steps"]
    return got

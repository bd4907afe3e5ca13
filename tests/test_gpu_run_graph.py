"""Model.run's captured host-checked steps (integrators.RKIntegrator.device_step)
against the same run with eager launches (hipgraph off), bit for bit: states,
times and dt, every model, direct and iterative solvers, parameters changed
and meshes re-finalised between runs, and the solver's check of every step."""
import numpy as np
import pytest
import torch

from test_gpu_euler import _device
from helpers import random_mask

pytestmark = pytest.mark.gpu


def _start(model, nx, ny, nisl, precision, hipgraph, dt=0.0, **kw):
    p = dict(model=model, nx=nx, ny=ny, Lx=nx / ny, Ly=1.0, tend=1e9, maxite=11, dt=dt,
             nprint=10 ** 9, hipgraph=hipgraph, **kw)
    msk = random_mask(ny, nx, 6, p.get("xperiodic", False), False, nisl=nisl) if nisl else None
    m = _device(p, msk, precision)
    rng = np.random.default_rng(3)
    x, y = m.mesh.xy("c")
    w = (np.exp(-((x - 0.5 * nx / ny) ** 2 + (y - 0.5) ** 2) / 0.02)
         + 1e-2 * rng.standard_normal(x.shape)) * m.mesh.msk * m.mesh.area
    s = m.state
    if model == "euler":
        s.u.x[...] = w * m.mesh.mskx
        s.u.y[...] = -w * m.mesh.msky
    elif model in ("rsw", "qgrsw"):
        s.h[...] = (m.mesh.area * m.mesh.msk + 0.05 * w)
    else:
        getattr(s, {"qg": "pv", "advection": "q"}.get(model, "omega"))[...] = w
    if model == "advection":
        s.U.x[...] = 0.3 * m.mesh.mskx / m.mesh.dx
    if kw.get("beta"):
        m.mesh.f = 0.1 * np.broadcast_to(y, x.shape) * m.mesh.area
    m.mesh.fill(s[0])
    m.integrator.diag(s)
    return m


def _leaves(m):
    out = []
    for v in m.state:
        out += list(v) if isinstance(v, tuple) else [v]
    return out


@pytest.mark.parametrize("model,nx,ny,nisl,precision,kw", [
    ("euler", 40, 40, 0, "fp64", {}), ("euler", 48, 40, 3, "fp64", {}),
    ("euler", 64, 64, 0, "fp32", {}),
    ("eulerpsi", 64, 64, 0, "fp64", {}), ("eulerpsi", 48, 40, 0, "fp32", dict(xperiodic=True)),
    ("eulerpsi", 64, 64, 0, "fp32", dict(xperiodic=True, yperiodic=True)),
    ("eulerpsi", 64, 64, 3, "fp64", dict(dt=0.01)),
    ("eulerpsi", 40, 40, 0, "fp64", dict(poisson_solver="mg")),
    ("qg", 64, 48, 0, "fp64", dict(beta=1.0, f0=5.0)), ("qgrsw", 64, 64, 1, "fp32", dict(dtmax=0.02)),
    ("rsw", 50, 40, 3, "fp64", {}), ("advection", 50, 40, 0, "fp64", {})])
def test_run_replays_match_eager(dev, model, nx, ny, nisl, precision, kw):
    print(f"\nrun {model} {nx}x{ny} islands={nisl} {precision} {kw}", flush=True)
    a, b = (_start(model, nx, ny, nisl, precision, g, **kw) for g in (True, False))
    for k in range(3):
        if k == 1:  # the next runs bake another CFL number
            for m in (a, b):
                m.param.cfl = 0.7
        if k == 2:
            for m in (a, b):
                m.mesh.finalize()
                m.integrator.diag(m.state)
        for m in (a, b):
            m.time.ite0, m.param.maxite = m.time.ite, 11 + k
            m.run()
        assert a.time.ite == b.time.ite and a.time.t == b.time.t and a.time.dt == b.time.dt
        for u, v in zip(_leaves(a), _leaves(b)):
            assert np.array_equal(u, v, equal_nan=True)
    captured = len(a.integrator._checked)
    direct = kw.get("poisson_solver") != "mg" and not (model == "euler" and nisl)
    assert (captured > 0) == direct and not b.integrator._checked
    for e, f in zip(a.integrator._solvers(), b.integrator._solvers()):
        if direct:
            assert e.read_stats()["solves"] == f.read_stats()["solves"] and e.calls == f.calls


def test_replayed_steps_are_checked(dev, monkeypatch):
    """A solve whose residual is not accepted ends the run with
    PoissonNotConverged, replayed or not, and does not linger."""
    from fluids2d_amd.elliptic import PoissonNotConverged
    m = _start("eulerpsi", 64, 64, 0, "fp64", True)
    m.run()
    assert m.integrator._checked
    pois = m.mesh.poisson_vertices
    with monkeypatch.context() as mp:
        mp.setattr(type(pois), "_accepted", lambda self, r: r <= 1e-30)
        m.time.ite0 = m.time.ite
        with pytest.raises(PoissonNotConverged):
            m.run()
    m.time.ite0 = m.time.ite
    m.run()


def test_planetary_vorticity_rebound_between_steps(dev):
    """qg with beta: mesh.f bound to another array during a run reaches the
    replayed steps, as it does the eager ones."""
    out = []
    for g in (True, False):
        m = _start("qg", 64, 64, 0, "fp64", g, beta=1.0)

        def rebind():
            if m.time.ite == 6:
                m.mesh.f = 3.0 * m.mesh.f
        rebind.device = True
        rebind.finalize = lambda: None
        m.diags.append(rebind)
        m.run()
        out.append(m.state.pv.copy())
    assert np.array_equal(*out)


@pytest.mark.parametrize("precision,change", [
    ("fp64", lambda m: setattr(m.param, "integrator", "enrk3")),
    ("fp64", lambda m: setattr(m.param, "compflux", "centered")),
    ("fp32", lambda m: m.mesh.poisson_vertices.set_refine(0))])
def test_changes_between_runs_reach_replayed_steps(dev, precision, change):
    """What an eager stage reads at every call -- the integrator's
    coefficients, the flux method, the refinements of a solve -- is not kept
    from an earlier run's graph."""
    out = []
    for g in (True, False):
        m = _start("eulerpsi", 64, 64, 0, precision, g, poisson_refine="every")
        m.run()
        before = m.state.omega.copy()
        change(m)
        m.time.ite0 = m.time.ite
        m.run()
        out.append(m.state.omega.copy())
    assert np.array_equal(*out) and not np.array_equal(out[0], before)


class _Reads:
    """A Param that notes the names read from it."""

    def __init__(self, param, names):
        self.__dict__.update(_param=param, _names=names)

    def __getattr__(self, name):
        self._names.add(name)
        return getattr(self._param, name)

    def __setattr__(self, name, value):
        setattr(self._param, name, value)


@pytest.mark.parametrize("model,precision,kw", [
    ("euler", "fp64", {}), ("eulerpsi", "fp64", {}), ("eulerpsi", "fp32", {}),
    ("qg", "fp64", dict(beta=1.0)), ("qgrsw", "fp32", dict(dtmax=0.02)), ("rsw", "fp64", {}),
    ("advection", "fp64", {})])
def test_captured_steps_read_keyed_parameters_only(dev, model, precision, kw):
    """Every parameter read while a step is captured is part of its key."""
    m = _start(model, 64, 64, 0, precision, True, **kw)
    m.run()
    integ, names = m.integrator, set()
    integ._checked.clear()
    integ.begin(m.state)
    integ.set_dt(m.time)
    for o in (integ, integ.model, m.mesh):
        o.param = _Reads(o.param, names)
    if integ._wants_dtn():
        integ._dtn_valid = True
    integ._pays = lambda time: True  # (reads the run's length)
    names.clear()
    assert integ._checked_step(m.time) is not None
    assert "integrator" in names and names <= set(integ.BAKED) | {"dt"}, names


@pytest.mark.parametrize("model,kw", [("qg", dict(beta=1.0)), ("euler", {}), ("advection", {}),
                                      ("qgrsw", dict(dtmax=0.02)), ("eulerpsi", {})])
def test_captured_steps_own_their_reductions(dev, monkeypatch, model, kw):
    """A captured step (of a run, or of device_steps) forms the CFL step in
    arrays of its model, not in the library's scratch of the stream it was
    captured on: that is another stream's, or another model's to grow."""
    from fluids2d_amd import _lib, operators
    made = []
    plain = _lib.call

    def call(name, *args):
        if torch.cuda.is_current_stream_capturing():
            made.append((name, args))
        return plain(name, *args)
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(operators, "call", call)
    m = _start(model, 64, 64, 0, "fp64", True, **kw)
    m.param.maxite = 40
    m.run()
    m.integrator.begin(m.state)
    m.integrator.device_steps(12)
    assert m.integrator._checked and m.integrator.graph_count()
    assert any(n.startswith(("f2d_cfl", "f2d_perpgrad_part")) for n, _ in made)
    for name, args in made:
        assert name != "f2d_cfl_dt"
        assert name != "f2d_perpgrad_ex" or args[10:12] == (None, None)


def test_captured_step_outlives_larger_reductions(dev):
    """The library's reduction scratch grows (its old allocation freed) for a
    grid of more blocks than the smallest allocation holds, between two runs
    of a captured model."""
    from fluids2d_amd import _lib
    n = 2920  # 4 points a thread of 256: 8360 blocks, 8192 is the smallest
    out = []
    for g in (True, False):
        m = _start("qg", 64, 64, 0, "fp64", g, beta=1.0)
        m.run()
        if g:
            assert m.integrator._checked
            param = type(m.param)()
            param.nx = param.ny = n
            grid = _lib.make_grid(param)
            a = [torch.zeros(n + 6, n + 6, dtype=torch.float32, device=dev) for _ in range(3)]
            msk = torch.ones(n + 6, n + 6, dtype=torch.int8, device=dev)
            dt = torch.zeros(1, dtype=torch.float64, device=dev)
            _lib.call("f2d_perpgrad_ex", _lib.F32, grid, *map(_lib.ptr, a), _lib.ptr(msk),
                      _lib.ptr(msk), 1.0, 1.0, 0, None, _lib.ptr(dt), 0.5, 2.0,
                      _lib.stream_ptr())
            assert float(dt) == 2.0
        m.time.ite0 = m.time.ite
        m.run()
        out.append(m.state.pv.copy())
    assert np.array_equal(*out)


@pytest.mark.parametrize("graph", [True, False])
def test_rejected_step_is_not_pushed_forward(dev, monkeypatch, graph):
    """The exception of a solve that is not accepted comes from its own step:
    the time stays where it was and no diagnostic sees the step."""
    from fluids2d_amd.elliptic import PoissonNotConverged
    m = _start("eulerpsi", 64, 64, 0, "fp64", graph)
    m.run()
    seen = []
    diag = lambda: seen.append(m.time.ite)  # noqa: E731
    diag.device, diag.finalize = True, lambda: None
    m.diags.append(diag)
    monkeypatch.setattr(type(m.mesh.poisson_vertices), "_accepted", lambda self, r: r <= 1e-30)
    m.time.ite0 = ite = m.time.ite
    t = m.time.t
    with pytest.raises(PoissonNotConverged):
        m.run()
    assert m.time.ite == ite and m.time.t == t and not seen


def test_resident_steps_after_replayed_ones(dev):
    """device_steps may capture its own graph right after a replayed
    device_step."""
    out = []
    for g in (True, False):
        m = _start("eulerpsi", 64, 64, 0, "fp64", g)
        integ = m.integrator
        integ.begin(m.state)
        dts = []
        for n in (16, 3, 8, 1, 8):
            if n % 8:
                for _ in range(n):
                    integ.set_dt(m.time)
                    integ.device_step(m.time)
                    dts.append(m.time.dt)
            else:
                dts += integ.device_steps(n).cpu().tolist()
        integ.end(m.state)
        out.append((m.state.omega.copy(), dts))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]



@pytest.mark.parametrize("model,kw,short,long", [
    ("eulerpsi", {}, dict(maxite=8), dict(maxite=30)),
    ("eulerpsi", dict(dt=0.01), dict(tend=0.05), dict(tend=0.4)),
    ("rsw", {}, dict(maxite=24), dict(maxite=60))])
def test_short_runs_capture_nothing(dev, model, kw, short, long):
    """A capture costs what some ten replayed steps save: a run with fewer
    steps to come, by maxite or by tend, stays eager, its first and (while all
    its runs together are short) its later ones."""
    m = _start(model, 64, 64, 0, "fp64", True, **kw)
    m.param.maxite = 10 ** 6
    for k, v in short.items():
        setattr(m.param, k, v)
    m.run()
    integ = m.integrator
    assert m.time.ite > 3 and not integ._checked
    n = m.time.ite
    for k, v in long.items():
        setattr(m.param, k, v)
    m.time.ite0, m.time.t0 = m.time.ite, m.time.t
    m.run()
    assert m.time.ite > n and integ._checked

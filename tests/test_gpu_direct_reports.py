"""What direct elliptic solves report: a right-hand side that is not finite
(csrc: k_fft_stats, k_cap_stats, k_modal_stats) on every route, to the caller
and in the device statistics."""
import math

import numpy as np
import pytest
import torch

from helpers import random_mask

pytestmark = pytest.mark.gpu


def _solver(nx, ny, nisl=0, precision="fp64", location="v", **kw):
    import fluids2d_amd.param as fp
    from fluids2d_amd import Model, Param
    fp.QUIET = True
    p = Param()
    for k, v in dict(model="euler" if location == "c" else "eulerpsi", nx=nx, ny=ny,
                     Lx=nx / 64.0, Ly=ny / 64.0, precision=precision, **kw).items():
        setattr(p, k, v)
    m = Model(p)
    if nisl:
        m.mesh.msk[...] = random_mask(ny, nx, 6, p.xperiodic, p.yperiodic, nisl=nisl)
        m.mesh.finalize()
    return m.mesh.poisson_vertices if location == "v" else m.mesh.poisson_centers


ROUTES = [
    ("fft", dict(nx=64, ny=64)), ("fft", dict(nx=64, ny=64, precision="fp32")),
    ("fft", dict(nx=64, ny=128, xperiodic=True, yperiodic=True)),
    ("fft", dict(nx=64, ny=64, location="c")),
    ("capacitance", dict(nx=64, ny=64, nisl=3)),
    ("capacitance", dict(nx=64, ny=64, nisl=3, precision="fp32")),
    ("modal", dict(nx=40, ny=48)), ("modal", dict(nx=40, ny=48, precision="fp32")),
    ("modal", dict(nx=40, ny=48, location="c")),
    ("modal_capacitance", dict(nx=40, ny=48, nisl=3)),
    ("modal_capacitance", dict(nx=40, ny=48, nisl=3, precision="fp32"))]


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("method,kw", ROUTES)
def test_solves_that_are_not_finite_are_reported(dev, method, kw, bad):
    from fluids2d_amd.elliptic import PoissonNotConverged
    ps = _solver(**kw)
    assert ps.method == method
    wet = ps.msk != 0
    b = np.random.default_rng(2).standard_normal(ps.msk.shape) * wet
    if method == "fft" or kw.get("location") == "c":
        b[wet] -= b[wet].mean()
    good = torch.from_numpy(b).to(dev, ps.dtype)
    spoilt = good.clone()
    spoilt[tuple(np.argwhere(wet)[0])] = bad
    ps.reset_stats()
    ps.solve(spoilt, torch.zeros_like(good), check=False)
    assert math.isnan(ps.last_relres)
    st = ps.read_stats()
    assert st["solves"] == 1 and st["failed"] == 1 and math.isnan(st["last_relres"])
    ps.solve(good, torch.zeros_like(good))
    assert ps.last_relres <= 1e-4
    stats = ps._stats_host()
    # (the device's own flag is set at 1e-6, FP32 storage can stay above it)
    assert stats[2] == (ps.last_relres <= 1e-6) and stats[4] == 2 - stats[2]
    assert math.isnan(stats[7])  # kept
    ps.reset_stats()
    ps.solve(good, torch.zeros_like(good))
    assert ps._stats_host()[7] == ps.last_relres
    # raised where multigrid raised it; on the other routes a run goes on to
    # its own check for values that are not finite, which stops it cleanly
    if method.startswith("modal"):
        with pytest.raises(PoissonNotConverged):
            ps.solve(spoilt, torch.zeros_like(good))
    else:
        ps.solve(spoilt, torch.zeros_like(good))


@pytest.mark.parametrize("nx,ny,nisl", [(64, 64, 3), (64, 64, 0)])
def test_spoilt_run_stops_cleanly(dev, nx, ny, nisl):
    """A NaN in the state of a run on these routes, eager or replayed, ends at
    the next synchronisation point with the state copied back."""
    import fluids2d_amd.param as fp
    from fluids2d_amd import Model, Param
    fp.QUIET = True
    for graph in (True, False):
        p = Param()
        for k, v in dict(model="eulerpsi", nx=nx, ny=ny, tend=1e9, maxite=24, nprint=10 ** 9,
                         hipgraph=graph).items():
            setattr(p, k, v)
        m = Model(p)
        if nisl:
            m.mesh.msk[...] = random_mask(ny, nx, 6, nisl=nisl)
            m.mesh.finalize()
        x, y = m.mesh.xy("c")
        m.state.omega[...] = np.exp(-((x - 0.5) ** 2 + (y - 0.5) ** 2) / 0.02) * m.mesh.msk \
            * m.mesh.area
        m.integrator.diag(m.state)

        def spoil():
            if m.time.ite == 18:
                j, i = np.argwhere(m.mesh.msk[3:-3, 3:-3])[7] + 3
                m.integrator.dstate.omega[j, i] = float("nan")
        spoil.device = True
        spoil.finalize = lambda: None
        m.diags.append(spoil)
        m.run()
        assert m.nonfinite == ["omega"] and m.time.ite == 24


def _condition(nx, ny, xper=False, yper=False, lx=1.0, ly=1.0, maindiag=0.0, cells=False):
    """Condition number of the rectangle's operator from its eigenvalues, on
    the zero-mean functions where it is singular."""
    def lam(n, per, c):
        k = np.arange(n) if per or cells else np.arange(1, n)
        return 4 * c * np.sin((np.pi if per else np.pi / 2) * k / n) ** 2
    dx, dy = lx / nx, ly / ny
    v = (lam(nx, xper, dy / dx)[:, None] + lam(ny, yper, dx / dy) + maindiag).ravel()
    return v.max() / v[v > 1e-13 * v.max()].min()


@pytest.mark.parametrize("method,kw,factor", [
    ("modal", dict(nx=40, ny=48), 64), ("modal", dict(nx=9, ny=8, precision="fp32"), 64),
    ("modal", dict(nx=300, ny=65, xperiodic=True), 64),
    ("modal", dict(nx=61, ny=30, yperiodic=True, location="c"), 64),
    ("modal", dict(nx=40, ny=41, xperiodic=True, yperiodic=True), 64),
    ("modal_capacitance", dict(nx=40, ny=48, nisl=3), 64),
    ("fft", dict(nx=4096, ny=64, xperiodic=True, yperiodic=True), 64),
    ("fft", dict(nx=64, ny=64), None), ("fft", dict(nx=64, ny=64, precision="fp32"), None),
    ("capacitance", dict(nx=64, ny=64, nisl=3), None), ("mg", dict(nx=40, ny=48), 0)])
def test_acceptance(dev, method, kw, factor):
    """A direct solve that takes the place of an iteration to rtol is accepted
    at rtol or at the bound of its rounding; a smooth right-hand side, whose
    solution is the largest, stays inside; the other routes' tests stay."""
    kw = dict(kw)
    if method == "mg":
        kw["poisson_solver"] = "mg"
    ps = _solver(**kw)
    assert ps.method == method
    single = kw.get("precision") == "fp32"
    if factor is None:
        assert ps.accept() == (1e-4 if single else 1e-6)
        ps.rtol = 1e-2
        assert ps.accept() == (1e-4 if single else 1e-6)
        return
    geo = {k: v for k, v in kw.items() if k in ("nx", "ny")}
    cond = _condition(**geo, xper=kw.get("xperiodic", False), yper=kw.get("yperiodic", False),
                      lx=kw["nx"] / 64.0, ly=kw["ny"] / 64.0, cells=kw.get("location") == "c")
    bound = factor * 2.0 ** -53 * (cond + 100)
    assert ps.accept() == pytest.approx(max(ps.rtol, bound), rel=1e-6)
    if method != "mg":
        assert bound < 5e-8  # not the 1e-6 of the other routes
    wet = ps.msk != 0
    j, i = np.mgrid[0:wet.shape[0], 0:wet.shape[1]]
    b = np.cos(2 * np.pi * (i - 3) / kw["nx"]) * np.cos(np.pi * (j - 3) / kw["ny"]) * wet
    if kw.get("location") == "c" or kw.get("yperiodic"):
        b[wet] -= b[wet].mean()
    x = torch.zeros(b.shape, dtype=ps.dtype, device=dev)
    ps.reset_stats()
    ps.solve(torch.from_numpy(b).to(dev, ps.dtype), x)
    st = ps.read_stats()
    assert st["failed"] == 0 and ps.last_relres <= ps.accept()
    assert not ps._accepted(1e-7)
    ps.rtol = 1e-3  # a looser one is the caller's to choose
    assert ps._accepted(9e-4) and not ps._accepted(2e-3)


@pytest.mark.parametrize("method,kw", [r for r in ROUTES if "location" not in r[1]])
def test_measured_solves_capture(dev, method, kw):
    """A measured solve allocates nothing: the first of a handle may be
    captured, and each replay measures what it solved."""
    from fluids2d_amd import _lib
    ps = _solver(**kw)
    assert ps.method == method
    wet = ps.msk != 0
    rng = np.random.default_rng(4)
    b, x = (torch.zeros(wet.shape, dtype=ps.dtype, device=dev) for _ in range(2))
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with _lib.capture(g):
        x.zero_()
        ps.solve(b, x, stats="device")
    for _ in range(3):
        w = rng.standard_normal(wet.shape) * wet
        w[wet] -= w[wet].mean()
        b.copy_(torch.from_numpy(w))
        ps.reset_stats()
        g.replay()
        got = x.clone()
        st = ps._stats_host()
        assert st[6] == 1 and 0.0 < st[1] == st[7] <= ps.accept()
        want = torch.zeros_like(x)
        ps.solve(b, want)
        err = (got - want).double().norm() / want.double().norm()
        assert err <= (1e-5 if ps.dtype == torch.float32 else 1e-12)

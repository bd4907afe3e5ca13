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

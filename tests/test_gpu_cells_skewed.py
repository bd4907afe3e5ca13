"""All-wet Neumann cell operators on long, thin rectangles: the direct solves
need no multigrid hierarchy, whose coarsest level such sizes make too long."""
import numpy as np
import pytest
import torch

from test_gpu_direct_reports import _solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,per,method", [
    (1200, 8, False, "modal"), (8, 1200, False, "modal"), (4000, 9, True, "modal"),
    (3, 40, False, "neumann"), (4096, 8, True, "fft"), (40, 40, False, "modal")])
def test_long_thin_rectangles(dev, nx, ny, per, method):
    from fluids2d_amd._lib import F2DError
    ps = _solver(nx=nx, ny=ny, xperiodic=per, yperiodic=per, location="c")
    assert ps.method == method
    wet = ps.msk != 0
    b = np.random.default_rng(nx).standard_normal(wet.shape) * wet
    b[wet] -= b[wet].mean()
    x = torch.zeros(b.shape, dtype=torch.float64, device=dev)
    ps.solve(torch.from_numpy(b).to(dev), x)
    u = np.pad(x.cpu().numpy()[3:-3, 3:-3], 1, mode="wrap" if per else "edge")
    r = u[1:-1, 2:] + u[1:-1, :-2] + u[2:, 1:-1] + u[:-2, 1:-1] - 4 * u[1:-1, 1:-1] \
        - b[3:-3, 3:-3]
    # as the solve itself measures it
    assert np.linalg.norm(r) <= 2 * ps.accept() * np.linalg.norm(b)
    with pytest.raises(F2DError):  # no multigrid kernels to time
        ps.bench_kernel(0)

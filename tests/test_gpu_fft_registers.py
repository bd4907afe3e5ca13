"""Spectral solves whose passes run as register transforms
(csrc/f2d_fft.hip): every length that takes them, beside a short other
direction, by the residual of the operator computed in numpy."""
import math

import numpy as np
import pytest
import torch

from test_gpu_kernels import N, T

pytestmark = pytest.mark.gpu

CASES = [(ny, 64, "fp64", True, True) for ny in (128, 256, 512, 1024, 2048, 4096)] + \
        [(512, 16, "fp64", True, False), (512, 64, "fp64", False, False),
         (1024, 32, "fp64", True, False), (64, 2048, "fp64", True, True),
         (64, 2048, "fp64", True, False), (16, 1024, "fp64", False, False),
         (2048, 64, "fp32", True, True), (4096, 64, "fp32", True, True),
         (1024, 64, "fp32", True, False), (1024, 64, "fp32", False, False),
         (2048, 64, "fp32", False, False), (64, 2048, "fp32", True, True),
         (64, 4096, "fp32", True, True), (16, 1024, "fp32", False, False),
         (64, 2048, "fp32", False, False)]


@pytest.mark.parametrize("ny,nx,precision,xper,yper", CASES)
def test_register_transforms(dev, ny, nx, precision, xper, yper):
    import fluids2d_amd.param as fp
    from fluids2d_amd import Model, Param
    fp.QUIET = True
    # square cells
    p = Param()
    for k, v in dict(model="eulerpsi", nx=nx, ny=ny, xperiodic=xper, yperiodic=yper,
                     precision=precision, poisson_warm=False, Lx=nx / 16.0,
                     Ly=ny / 16.0).items():
        setattr(p, k, v)
    ps = Model(p).mesh.poisson_vertices
    assert ps.method == "fft"
    ys, xs = slice(0 if yper else 1, ny), slice(0 if xper else 1, nx)  # unknowns
    w = np.zeros((ny, nx))
    w[ys, xs] = np.random.default_rng(nx + ny).standard_normal(w[ys, xs].shape)
    if xper and yper:
        w -= w.mean()
    w = w.astype("f4" if precision == "fp32" else "f8").astype(float)  # (representable)
    b = np.zeros((ny + 6, nx + 6))
    b[3:-3, 3:-3] = w

    def residual(x):
        u = np.zeros((ny + 2, nx + 2))
        u[1:-1, 1:-1][ys, xs] = x[3:-3, 3:-3][ys, xs]
        if xper:
            u[:, 0], u[:, -1] = u[:, -2], u[:, 1]
        if yper:
            u[0], u[-1] = u[-2], u[1]
        a = u[1:-1, 2:] + u[1:-1, :-2] + u[2:, 1:-1] + u[:-2, 1:-1] - 4 * u[1:-1, 1:-1]
        r = (a - w)[ys, xs]
        return np.linalg.norm(r - (r.mean() if xper and yper else 0.0)), np.linalg.norm(u)

    bt = T(b, dev).to(ps.dtype)
    x = torch.zeros(b.shape, dtype=ps.dtype, device=dev)
    if precision == "fp32":
        ps.set_refine(0)
    ps.solve(bt, x, check=False)
    r, nu = residual(N(x).astype(float))
    # two forward and two inverse transforms, ||A|| = 8: the rounding of x's
    # spectrum (and of x itself, FP32) through the operator
    eps = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    bound = 8 * nu * eps * 4 * math.log2(nx * ny)
    print(f"\n{ny}x{nx} {precision} residual {r:.2e} bound {bound:.2e}")
    assert r <= bound
    if precision == "fp32":
        # a refinement in FP64 takes the FP32 solve's residual down by FP32
        # rounding times the digits that the operator loses between the
        # lowest and the other modes of a residual (some 100)
        ps.set_refine(1)
        ps.solve(bt, x)
        ratio = ps.last_relres * np.linalg.norm(w) / r
        print(f"  refined relres {ps.last_relres:.2e} contraction {ratio:.1e}")
        assert ratio <= 100 * eps * math.log2(nx * ny)

"""The capacitance solve with few and many boundary points (one tile of M up
to more tile rows than the waves of the sum of its partials), and with NaN in
the right-hand side outside the unknowns, which the fused masks must drop."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import P
from test_gpu_capacitance import _handle, _solve, L  # noqa: F401  (L: a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["f64", "refine"])
@pytest.mark.parametrize("every,rows", [(128, 1), (16, 4), (7, 21)])
def test_boundary_sizes(dev, L, every, rows, mode):  # noqa: F811
    n = 128
    p = P(model="eulerpsi", nx=n, ny=n, xperiodic=True, yperiodic=False, Lx=2.0, Ly=1.6)
    m = np.zeros((n + 6, n + 6), dtype=np.int8)
    m[3:-3, 3:-3] = 1
    m[7:-7:every, 7:-7:every] = 0  # single dry cells
    O.fill(p, m)
    mesh = O.Mesh(p, msk=m)
    unk = O.unknown_mask(p, mesh.mskv)
    wet = (unk != 0)
    rect = np.zeros_like(wet)
    rect[4:-3, 3:-3] = True
    near = np.zeros_like(wet)  # rectangle unknowns that are dry beside a wet one
    for ax in (0, 1):
        for s in (-1, 1):
            near |= np.roll(wet, s, ax)
    assert -(-int((rect & ~wet & near).sum()) // 64) == rows
    b = np.random.default_rng(5).standard_normal(m.shape) * mesh.mskv
    ref = np.zeros(m.shape)
    O.Poisson2D(p, mesh, "v").solve(b, ref)
    b[3:-3, 3:-3][~wet[3:-3, 3:-3]] = np.nan
    h = _handle(L, unk, p, 0.0, L.POISSON_F64 if mode == "f64" else L.POISSON_F32_REFINE)
    assert L.lib().f2d_poisson_method(h) == L.SOLVERS["cap"]
    dt = torch.float64 if mode == "f64" else torch.float32
    x = torch.zeros(m.shape, dtype=dt, device=dev)
    it, rr = _solve(L, h, torch.from_numpy(b).to(dev, dt), x, False)
    L.call("f2d_poisson_destroy", h)
    err = np.linalg.norm(x.double().cpu().numpy() - ref) / np.linalg.norm(ref)
    print(f"\nevery {every} {mode}: relres={rr:.2e} err={err:.2e}")
    # FP64: the bars of the solves against SuperLU.  FP32: one refinement
    # squares the FP32 solve's relative residual, rounding times the condition
    # of C (logarithmic interactions of |B| points: O(|B|))
    assert rr <= (1e-12 if mode == "f64" else (8 * 64 * rows * 2.0 ** -24) ** 2)
    assert err <= (1e-11 if mode == "f64" else 1e-7)

"""The masked Neumann cell operator (csrc/f2d_neumann.hip) by CG with the
rectangle's direct solve as preconditioner, against SuperLU (the oracle's
Poisson2D): islands, a basin that leaves most of the rectangle dry, two
regions behind a one-cell wall, periodic directions, FP64 and FP32 storage,
eigenvector and FFT rectangles, a right-hand side of an earlier NaN solve."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from helpers import P, random_mask
from test_gpu_kernels import L, N, T  # noqa: F401  (L: a fixture)

pytestmark = pytest.mark.gpu


def _mask(kind, ny, nx, xper, yper):
    if kind == "islands":
        return random_mask(ny, nx, 5, xper, yper, nisl=5)
    m = O.default_mask(ny, nx, 3, xper, yper)
    jj, ii = np.mgrid[0:ny + 6, 0:nx + 6]
    if kind == "basin":
        m[((jj - 3 - ny / 2) / ny) ** 2 + ((ii - 3 - nx / 2) / nx) ** 2 > 0.16] = 0
    else:  # a wall one cell thick: two regions, each with its own constant
        m[:, 3 + nx // 3] = 0
    return m


def _regions(unk, xper, yper):
    """Labels of the connected unknowns (4 neighbours, periodic wrap)."""
    from scipy import ndimage
    lab, _ = ndimage.label(unk[3:-3, 3:-3])
    for per, a, b in ((xper, lab[:, 0], lab[:, -1]), (yper, lab[0], lab[-1])):
        if per:
            for u, v in zip(a, b):
                if u and v and u != v:
                    a_, b_ = max(u, v), min(u, v)
                    lab[lab == a_] = b_
    return lab


@pytest.mark.parametrize("ny,nx,xper,yper,kind,maindiag,single", [
    (40, 48, False, False, "islands", 0.0, False), (64, 64, False, False, "basin", 0.0, False),
    (33, 90, True, False, "islands", 0.0, False), (50, 41, False, True, "islands", 0.0, False),
    (60, 61, True, True, "islands", 0.0, False), (48, 64, False, False, "wall", 0.0, False),
    (64, 33, False, False, "islands", 0.2, False), (40, 48, False, False, "basin", 0.0, True),
    (512, 512, False, False, "islands", 0.0, False)])
def test_masked_cells_vs_superlu(dev, L, ny, nx, xper, yper, kind, maindiag, single):
    p = P(model="euler", nx=nx, ny=ny, xperiodic=xper, yperiodic=yper, Lx=nx / 64.0,
          Ly=ny / 70.0)
    mesh = O.Mesh(p, msk=_mask(kind, ny, nx, xper, yper))
    unk = O.unknown_mask(p, mesh.msk)
    lab = _regions(unk, xper, yper)
    inner = np.zeros(unk.shape, dtype=np.int64)
    inner[3:-3, 3:-3] = lab
    dt = torch.float32 if single else torch.float64
    rng = np.random.default_rng(1)
    b = N(T(rng.standard_normal(unk.shape) * unk, dev).to(dt)).astype(np.float64)
    x0 = N(T(rng.standard_normal(unk.shape), dev).to(dt)).astype(np.float64)
    bref = b.copy()
    x_ref = np.zeros(unk.shape)
    ids = [k for k in np.unique(lab) if k]
    if maindiag == 0.0:
        for k in ids:
            bref[inner == k] -= bref[inner == k].mean()
    # one region at a time: SuperLU leaves each region's constant to rounding
    for k in ids:
        u = (inner == k).astype(np.int8)
        G, n = O.gindex(u)
        A = O.laplacian(G, n, mesh.dx, mesh.dy, maindiag, True, xper, yper, 3)
        idx = G > -1
        if maindiag == 0.0:
            sol = np.zeros(n)
            sol[:-1] = O.splinalg.splu(A[:-1, :-1].tocsc()).solve(bref[idx][:-1])
            # the constant of each region stays the initial guess's
            sol += x0[idx].mean() - sol.mean()
        else:
            sol = O.splinalg.splu(A).solve(bref[idx])
        x_ref[idx] = sol
    opts = L.PoissonOpts()
    opts.mode = L.POISSON_F32_REFINE if single else L.POISSON_F64
    opts.nu, opts.neumann = 2, 1
    h = ctypes.c_void_p()
    L.call("f2d_poisson_create", unk.ctypes.data_as(ctypes.c_void_p),
           ctypes.byref(L.make_grid(p)), maindiag, ctypes.byref(opts), ctypes.byref(h))
    try:
        assert L.lib().f2d_poisson_method(h) == 3
        it, rr = ctypes.c_int(), ctypes.c_double()

        def solve(rhs, start):
            x = T(start, dev).to(dt)
            L.call("f2d_poisson_solve", h, L.ptr(T(rhs, dev).to(dt)), L.ptr(x), 1e-12, 2000,
                   ctypes.byref(it), ctypes.byref(rr), L.stream_ptr())
            return N(x).astype(np.float64)
        bad = b.copy()
        bad[tuple(np.argwhere(unk == 1)[0])] = np.nan
        k0 = inner[tuple(np.argwhere(unk == 1)[0])]
        assert np.isnan(solve(bad, x0)[inner == k0]).all()  # and forgotten by the next solve
        x = solve(b, x0)
        iters = it.value
        again = solve(b, x)  # from the solution: nothing left to do
    finally:
        L.call("f2d_poisson_destroy", h)
    wet = unk == 1
    err = np.linalg.norm((x - x_ref)[wet]) / np.linalg.norm(x_ref[wet])
    print(f"\nmasked cells {ny}x{nx} {kind} xper={xper} yper={yper} md={maindiag} f32={single}: "
          f"{iters} iterations, relres={rr.value:.2e} err={err:.2e}; again {it.value}")
    # residual 1e-12 times the condition number of the smooth modes (SuperLU
    # itself 1e-11 on the singular operator at 512^2); FP32: x is stored so
    assert err <= (1e-6 if single else 1e-9)
    assert iters <= 60  # Jacobi: 150 to 2000 on these grids
    assert it.value <= (iters if single else 3)
    # dry entries untouched but for the periodic images
    dry = np.zeros_like(wet)
    dry[3:-3, 3:-3] = ~wet[3:-3, 3:-3]
    assert np.array_equal(x[dry], x0[dry])

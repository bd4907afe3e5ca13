"""The eigenvector solve of fully wet rectangles whose sizes are not powers
of two (csrc/f2d_modal.hip) against SuperLU (the oracle's Poisson2D): every
combination of closed and periodic directions at the edges of its 16 x 16
tiles and chunks of 32 contraction pairs (test_gpu_modal_tiles.py has the
larger tiles), odd and even point counts, with and without mass term, vertex
and cell operators, the fused centerstovertices right-hand side, FP64 and FP32
storage."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from helpers import P, random_mask
from test_gpu_kernels import L, N, T, _poisson_case  # noqa: F401  (L: a fixture)

pytestmark = pytest.mark.gpu

# tile and chunk edges: pairs of 32 / 33 / 64 / 65 points a side, the smallest
# sizes, more output tiles than one per CU (800 x 304, 1000 x 600), odd sizes
SIZES = [(8, 9), (11, 10), (33, 32), (65, 63), (40, 40), (130, 66), (61, 200)]


PERIODS = [(False, False), (True, False), (False, True), (True, True)]
FORMS = [(0.0, False, False), (0.3, True, False), (0.0, True, True)]


@pytest.mark.parametrize("ny,nx,xper,yper,maindiag,c2v,single", [
    (*n, *per, *form) for n in SIZES for per in PERIODS for form in FORMS] + [
    (304, 800, True, False, *FORMS[0]), (304, 800, False, False, *FORMS[2]),
    (600, 1000, False, True, *FORMS[1])])
def test_modal_vertices_vs_superlu(dev, L, ny, nx, xper, yper, maindiag, c2v, single):
    p = P(model="eulerpsi", nx=nx, ny=ny, xperiodic=xper, yperiodic=yper, Lx=nx / 64.0,
          Ly=ny / 80.0)
    m = O.default_mask(ny, nx, 3, xper, yper)
    mode = L.POISSON_F32_REFINE if single else L.POISSON_F64
    err, it, rr, x, xr, unk = _poisson_case(dev, L, p, m, maindiag, mode, solver="auto", c2v=c2v)
    print(f"\nmodal {ny}x{nx} xper={xper} yper={yper} md={maindiag} c2v={c2v} f32={single}: "
          f"relres={rr:.2e} err={err:.2e}")
    assert it == 1
    # rounding (2.2e-16; 6e-8 where b and x are stored in FP32) times the
    # condition number, below 0.5 max(n)^2 (anisotropy 1.6): the smooth part
    # of white noise sees far less of it
    assert err <= (2e-7 if single else 1e-11)
    assert rr <= 1e-11  # in FP32 that of the result before it is rounded
    inner = np.zeros_like(unk, dtype=bool)
    inner[3:-3, 3:-3] = True
    assert np.all(x[inner & (unk == 0)] == 0)
    xx = x.copy()
    O.fill(p, xx)
    assert np.array_equal(xx, x)


@pytest.mark.parametrize("ny,nx", SIZES + [(160, 192)])
@pytest.mark.parametrize("xper,yper,maindiag,single", [
    (False, False, 0.0, False), (True, False, 0.0, False), (False, True, 0.2, False),
    (True, True, 0.0, False), (False, False, 0.0, True)])
def test_modal_cells_vs_superlu(dev, L, ny, nx, xper, yper, maindiag, single):
    """The Neumann cell operator of an all-wet domain (elliptic.py:186-190);
    solutions of the singular operator compared without their means."""
    p = P(model="euler", nx=nx, ny=ny, xperiodic=xper, yperiodic=yper, Lx=nx / 64.0,
          Ly=ny / 80.0)
    mesh = O.Mesh(p, msk=O.default_mask(ny, nx, 3, xper, yper))
    unk = O.unknown_mask(p, mesh.msk)
    inner = unk == 1
    b = (np.random.default_rng(3).standard_normal(unk.shape) + 0.5) * unk
    dt = torch.float32 if single else torch.float64
    b = N(T(b, dev).to(dt)).astype(np.float64)
    bref = b.copy()
    if maindiag == 0.0:
        bref[inner] -= bref[inner].mean()
    x_ref = np.zeros(unk.shape)
    O.Poisson2D(p, mesh, "c", maindiag=maindiag).solve(bref, x_ref)
    opts = L.PoissonOpts()
    opts.mode = L.POISSON_F32_REFINE if single else L.POISSON_F64
    opts.nu, opts.neumann = 2, 1
    h = ctypes.c_void_p()
    L.call("f2d_poisson_create", unk.ctypes.data_as(ctypes.c_void_p),
           ctypes.byref(L.make_grid(p)), maindiag, ctypes.byref(opts), ctypes.byref(h))
    try:
        assert L.lib().f2d_poisson_method(h) == 5
        x = torch.zeros(unk.shape, dtype=dt, device=dev)
        it, rr = ctypes.c_int(), ctypes.c_double()
        L.call("f2d_poisson_solve", h, L.ptr(T(b, dev).to(dt)), L.ptr(x), 1e-13, 2000,
               ctypes.byref(it), ctypes.byref(rr), L.stream_ptr())
        got = N(x).astype(np.float64)[inner]
    finally:
        L.call("f2d_poisson_destroy", h)
    want = x_ref[inner]
    if maindiag == 0.0:
        got, want = got - got.mean(), want - want.mean()
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"\nmodal cells {ny}x{nx} xper={xper} yper={yper} md={maindiag} f32={single}: "
          f"relres={rr.value:.2e} err={err:.2e}")
    # SuperLU's own rounding on the singular operator: 1e-11 at 512^2
    assert err <= (2e-7 if single else 1e-10)


@pytest.mark.parametrize("ny,nx,solver,method", [(40, 48, "auto", 5), (40, 48, "mg", 1),
                                                 (64, 64, "auto", 2)])
def test_modal_selection(dev, L, ny, nx, solver, method):
    """Taken by "auto" only, and not where the FFT solve applies; an explicit
    "fft" on such sizes stays refused."""
    from fluids2d_amd._lib import F2DError
    p = P(model="eulerpsi", nx=nx, ny=ny)
    unk = O.unknown_mask(p, O.Mesh(p).mskv)

    def create(name):
        opts = L.PoissonOpts()
        opts.nu, opts.solver = 2, L.SOLVERS[name]
        h = ctypes.c_void_p()
        L.call("f2d_poisson_create", unk.ctypes.data_as(ctypes.c_void_p),
               ctypes.byref(L.make_grid(p)), 0.0, ctypes.byref(opts), ctypes.byref(h))
        got = L.lib().f2d_poisson_method(h)
        L.call("f2d_poisson_destroy", h)
        return got
    assert create(solver) == method
    if method == 5:
        with pytest.raises(F2DError):
            create("fft")


def _masked(ny, nx, xper, yper, kind):
    if kind == "islands":
        return random_mask(ny, nx, 7, xper, yper, nisl=6)
    m = O.default_mask(ny, nx, 3, xper, yper)
    jj, ii = np.mgrid[0:ny + 6, 0:nx + 6]
    m[((jj - 3 - ny / 2) / ny) ** 2 + ((ii - 3 - nx / 2) / nx) ** 2 > 0.16] = 0
    return m


@pytest.mark.parametrize("ny,nx,xper,yper,kind,maindiag,single,c2v", [
    (40, 48, False, False, "basin", 0.0, False, False), (61, 90, True, False, "islands", 0.0,
                                                         False, True),
    (100, 50, False, True, "islands", 0.3, False, False), (64, 65, True, True, "islands", 0.5,
                                                           False, True),
    (96, 64, False, False, "basin", 0.0, True, True), (130, 300, True, False, "islands", 0.0,
                                                       True, False),
    (360, 500, False, False, "basin", 0.0, False, True)])
def test_modal_capacitance_vs_superlu(dev, L, ny, nx, xper, yper, kind, maindiag, single, c2v):
    """Masks inside such rectangles: the capacitance solve around the
    eigenvector solve, FP64 inside for either storage."""
    p = P(model="eulerpsi", nx=nx, ny=ny, xperiodic=xper, yperiodic=yper, Lx=nx / 64.0,
          Ly=ny / 80.0)
    mesh = O.Mesh(p, msk=_masked(ny, nx, xper, yper, kind))
    unk = O.unknown_mask(p, mesh.mskv)
    dt = torch.float32 if single else torch.float64
    w = np.random.default_rng(3).standard_normal(unk.shape) * (mesh.msk if c2v else mesh.mskv)
    if c2v:
        O.fill(p, w)
    w = N(T(w, dev).to(dt)).astype(np.float64)
    b = w.copy()
    if c2v:
        O.centerstovertices(mesh, w, b)
    x_ref = np.zeros(unk.shape)
    O.Poisson2D(p, mesh, "v", maindiag=maindiag).solve(b, x_ref)
    opts = L.PoissonOpts()
    opts.mode = L.POISSON_F32_REFINE if single else L.POISSON_F64
    opts.nu = 2
    h = ctypes.c_void_p()
    L.call("f2d_poisson_create", unk.ctypes.data_as(ctypes.c_void_p),
           ctypes.byref(L.make_grid(p)), maindiag, ctypes.byref(opts), ctypes.byref(h))
    try:
        assert L.lib().f2d_poisson_method(h) == 6
        x = torch.full(unk.shape, 7.0, dtype=dt, device=dev)
        it, rr = ctypes.c_int(), ctypes.c_double()
        name = "f2d_poisson_solve_c2v" if c2v else "f2d_poisson_solve"

        def solve(rhs):
            L.call(name, h, L.ptr(T(rhs, dev).to(dt)), L.ptr(x), 1e-13, 100, ctypes.byref(it),
                   ctypes.byref(rr), L.stream_ptr())
        bad = w.copy()
        bad[tuple(np.argwhere(unk == 1)[0])] = np.nan
        solve(bad)
        assert not rr.value <= 1.0  # reported, as multigrid does
        solve(w)
        got = N(x).astype(np.float64)
    finally:
        L.call("f2d_poisson_destroy", h)
    wet = unk == 1
    err = np.linalg.norm((got - x_ref)[wet]) / np.linalg.norm(x_ref[wet])
    print(f"\nmodal capacitance {ny}x{nx} xper={xper} yper={yper} {kind} md={maindiag} "
          f"f32={single} c2v={c2v}: relres={rr.value:.2e} err={err:.2e}")
    # the bars of the spectral capacitance solve; FP32 stores x to 6e-8 and
    # averages b in FP32
    assert rr.value <= 1e-11 and err <= (3e-7 if single else 1e-11)
    dry = np.zeros_like(wet)
    dry[3:-3, 3:-3] = ~wet[3:-3, 3:-3]
    assert np.all(got[dry] == 7.0)
    full = got.copy()
    O.fill(p, full)
    assert np.array_equal(full, got)

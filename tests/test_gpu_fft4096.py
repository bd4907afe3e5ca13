"""FP64 FFT solves with a periodic direction of 4096 points (transformed in
place in LDS, csrc/f2d_fft.hip): against the DFT closed form and, for the
channel, by the residual; the two-buffer limit of explicit requests stays."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from helpers import P
from test_gpu_kernels import L, N, T  # noqa: F401  (L: a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nx,yper,maindiag,c2v", [
    (64, 4096, True, 0.0, False), (4096, 64, True, 0.4, True), (4096, 4096, True, 0.0, True),
    (64, 4096, False, 0.0, False)])
def test_fft_4096_fp64(dev, L, ny, nx, yper, maindiag, c2v):
    p = P(model="eulerpsi", nx=nx, ny=ny, xperiodic=True, yperiodic=yper, Lx=nx / 64.0,
          Ly=ny / 80.0)
    unk = O.unknown_mask(p, O.Mesh(p).mskv)
    g = L.make_grid(p)

    def create(solver):
        opts = L.PoissonOpts()
        opts.mode, opts.nu, opts.solver = L.POISSON_F64, 2, L.SOLVERS[solver]
        h = ctypes.c_void_p()
        L.call("f2d_poisson_create", unk.ctypes.data_as(ctypes.c_void_p), ctypes.byref(g),
               maindiag, ctypes.byref(opts), ctypes.byref(h))
        return h
    with pytest.raises(L.F2DError, match="FP64"):
        create("fft")
    h = create("auto")
    try:
        assert L.lib().f2d_poisson_method(h) == 2
        w = np.zeros(unk.shape)
        w[3:-3, 3:-3] = np.random.default_rng(4).standard_normal((ny, nx))
        O.fill(p, w)
        x = torch.zeros(unk.shape, dtype=torch.float64, device=dev)
        it, rr = ctypes.c_int(), ctypes.c_double()
        L.call("f2d_poisson_solve_c2v" if c2v else "f2d_poisson_solve", h, L.ptr(T(w, dev)),
               L.ptr(x), 1e-13, 10, ctypes.byref(it), ctypes.byref(rr), L.stream_ptr())
        got = N(x)
    finally:
        L.call("f2d_poisson_destroy", h)
    print(f"\nfft {ny}x{nx} yper={yper} md={maindiag} c2v={c2v}: relres={rr.value:.2e}")
    # rounding times the condition number: 3e-12 at 512^2, n^2
    assert rr.value <= 2e-10
    full = got.copy()
    O.fill(p, full)
    assert np.array_equal(full, got)
    if yper:
        b = w
        if c2v:
            b = 0.25 * (w + np.roll(w, 1, 0) + np.roll(w, 1, 1) + np.roll(np.roll(w, 1, 0), 1, 1))
        want = O.fft_poisson_periodic(b[3:-3, 3:-3], p.Lx / nx, p.Ly / ny, maindiag)
        err = np.linalg.norm(got[3:-3, 3:-3] - want) / np.linalg.norm(want)
        print(f"  err={err:.2e}")
        # the closed form's eigenvalue cos(2 pi / 4096) - 1 = -1.2e-6 carries
        # the rounding of a cosine near 1: 1.1e-16 / 1.2e-6
        assert err <= 1e-10

"""Masked Neumann solves made without a host check: iterations enqueued behind
the converged one return at once, the preconditioner's spectral passes too."""
import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from helpers import P
from test_gpu_kernels import L, T  # noqa: F401  (L: a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [512, 2048])
def test_iterations_after_convergence_return(dev, L, n):  # noqa: F811
    p = P(model="euler", nx=n, ny=n, xperiodic=True, yperiodic=True, Lx=1.0, Ly=1.0)
    m = O.default_mask(n, n, 3, True, True)
    m[n // 3:n // 3 + 20, n // 4:n // 4 + 30] = 0
    O.fill(p, m)
    mesh = O.Mesh(p, msk=m)
    unk = O.unknown_mask(p, mesh.msk)
    b = T(np.random.default_rng(3).standard_normal(unk.shape) * unk, dev)
    opts = L.PoissonOpts()
    opts.mode, opts.nu, opts.neumann = L.POISSON_F64, 2, 1
    h = ctypes.c_void_p()
    L.call("f2d_poisson_create", unk.ctypes.data_as(ctypes.c_void_p),
           ctypes.byref(L.make_grid(p)), 0.0, ctypes.byref(opts), ctypes.byref(h))
    try:
        assert L.lib().f2d_poisson_method(h) == 3

        def run(rtol, maxit, checked=False):
            x = torch.zeros_like(b)
            it, rr = ctypes.c_int(), ctypes.c_double()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            L.call("f2d_poisson_solve", h, L.ptr(b), L.ptr(x), rtol, maxit,
                   ctypes.byref(it) if checked else None, ctypes.byref(rr) if checked else None,
                   L.stream_ptr())
            e1.record()
            e1.synchronize()
            return x, e0.elapsed_time(e1), it.value

        want, _, it = run(1e-10, 400, True)
        assert 2 <= it <= 40
        got, _, _ = run(1e-10, 200)
        assert torch.equal(got, want)  # what the checked solve stopped at
        few, many = (min(run(1e-10, k)[1] for _ in range(3)) for k in (100, 300))
        idle = (many - few) / 200
        busy = min(run(0.0, 40)[1] for _ in range(3)) / 40
        print(f"\n{n}^2: {it} iterations, {busy * 1e3:.1f} us each, idle {idle * 1e3:.1f} us")
        if n == 2048:  # (launches alone take as long as the work on small grids)
            assert idle <= 0.2 * busy
    finally:
        L.call("f2d_poisson_destroy", h)

"""The eigenvector solve's larger tiles (csrc/f2d_modal_plan.hpp: 32 x 32 from
400 of them, 64 x 64 from 640), on ragged sides and on matrix pitches that end
in half a widest tile: manufactured sums of eigenvectors, the residual of noise
formed in numpy, halo images, FP64 and FP32 storage, vertices and cells, the
fused centerstovertices right-hand side, and masked writes."""
import numpy as np
import pytest
import torch

from test_gpu_kernels import N, T

pytestmark = pytest.mark.gpu


def _tiles(rows, pairs, b):
    return -(-rows // b) * -(-pairs // b)


def _tile(nx, ny):
    """The tile of a solve (both directions' passes; mirror pairs: half of the
    points)."""
    for b, least in ((64, 640), (32, 400)):
        if min(_tiles(ny, nx // 2, b), _tiles(nx, ny // 2, b)) >= least:
            return b
    return 16


def _solver(nx, ny, xper, yper, precision, cells, mask=None):
    import fluids2d_amd.param as fp
    from fluids2d_amd import Model, Param
    fp.QUIET = True
    p = Param()
    for k, v in dict(model="euler" if cells else "eulerpsi", nx=nx, ny=ny, xperiodic=xper,
                     yperiodic=yper, precision=precision, Lx=nx / 64.0, Ly=ny / 64.0).items():
        setattr(p, k, v)
    m = Model(p)
    if mask is not None:
        mask(m.mesh.msk)
        m.mesh.fill(m.mesh.msk)
        m.mesh.finalize()
    return m, (m.mesh.poisson_centers if cells else m.mesh.poisson_vertices)


def _lam(k, n, per):
    """Eigenvalues of a direction's second difference."""
    return -4 * np.sin((np.pi if per else np.pi / 2) * k / n) ** 2


def _modes(n, per, cells):
    """A few eigenvectors of a direction's second difference on the n grid
    points (0 at a wall's first one), with their eigenvalues.  Angles from
    reduced indices: a rounded angle of some thousand is off by 1e-13."""
    i = np.arange(n)
    if per:
        ks = [0, 1, 3, n // 3, n // 2]
        ang = [2 * np.pi * (k * i % n) / n for k in ks]
        v = [np.cos(a) + (np.sin(a) if 0 < 2 * k < n else 0) for k, a in zip(ks, ang)]
    elif cells:
        ks = [0, 1, 2, n // 2 + 1, n - 1]
        v = [np.cos(np.pi * (k * (2 * i + 1) % (4 * n)) / (2 * n)) for k in ks]
    else:
        ks = [1, 2, 5, n // 2, n - 1]
        v = [np.sin(np.pi * (k * i % (2 * n)) / n) for k in ks]
    return [(f, _lam(k, n, per)) for k, f in zip(ks, v)]


def _amplified(nx, ny, xper, yper, cells):
    """Root mean square of 1 / eigenvalue: what the solve makes of rounding
    errors that are independent from point to point."""
    k0x, k0y = int(not (xper or cells)), int(not (yper or cells))
    lam = _lam(np.arange(k0x, nx), nx, xper) + _lam(np.arange(k0y, ny), ny, yper)[:, None]
    lam = lam[lam < 0]
    return np.sqrt(np.mean(lam ** -2.0))


def _apply(u, xper, yper, cells, wet):
    """The 5-point operator of square cells on the grid's points."""
    v = np.pad(u, 1, mode="edge" if cells else "constant")
    if xper:
        v[1:-1, 0], v[1:-1, -1] = u[:, -1], u[:, 0]
    if yper:
        v[0, 1:-1], v[-1, 1:-1] = u[-1], u[0]
    a = v[1:-1, 2:] + v[1:-1, :-2] + v[2:, 1:-1] + v[:-2, 1:-1] - 4 * u
    return a * wet


CASES = [
    # 32 x 32: ragged sides, odd sizes, every kind of direction
    (1100, 1030, 32, False, False, "fp64", False), (1031, 1100, 32, True, False, "fp32", False),
    (1027, 1090, 32, False, False, "fp64", True), (1100, 1030, 32, True, True, "fp64", False),
    # 64 x 64: pitches of 32 mod 64 (3000: 1500 pairs), odd sizes
    (3000, 2000, 64, False, False, "fp64", False), (2600, 2600, 64, True, True, "fp64", True),
    (2500, 2431, 64, True, False, "fp32", False), (2431, 2500, 64, False, True, "fp64", False),
    (3000, 2000, 64, False, False, "fp64", True)]


@pytest.mark.parametrize("nx,ny,tile,xper,yper,precision,cells", CASES)
def test_tiles(dev, nx, ny, tile, xper, yper, precision, cells):
    assert _tile(nx - 1, ny - 1) == _tile(nx + 2, ny + 2) == tile
    m, ps = _solver(nx, ny, xper, yper, precision, cells)
    assert ps.method == "modal"
    wet = np.ones((ny, nx))
    if not cells:
        wet[:, 0] *= xper
        wet[0] *= yper
    singular = cells or (xper and yper)

    def solve(b, c2v=False):
        p = np.zeros((ny + 6, nx + 6))
        p[3:-3, 3:-3] = b
        if c2v:
            m.mesh.fill(p)
        x = torch.zeros(p.shape, dtype=ps.dtype, device=dev)
        (ps.solve_c2v if c2v else ps.solve)(T(p, dev).to(ps.dtype), x)
        got = N(x).astype(float)
        full = got.copy()
        m.mesh.fill(full)
        assert np.array_equal(full, got)
        assert not np.any(got[3:-3, 3:-3][wet == 0])
        return got[3:-3, 3:-3]

    eps, store = 2.0 ** -53, 2.0 ** -24 if precision == "fp32" else 0.0
    # four products of up to n / 2 terms: rounding errors that add up as in a
    # random walk, a relative error of x of their number's root, twice over
    grow = 2 * 4 * np.sqrt(max(nx, ny) / 2)
    want, b = np.zeros((ny, nx)), np.zeros((ny, nx))
    for (fx, lx), (fy, ly) in zip(_modes(nx, xper, cells), _modes(ny, yper, cells)[::-1]):
        if lx + ly != 0.0:
            want += np.outer(fy, fx)
            b += (lx + ly) * np.outer(fy, fx)
    got = solve(b * wet)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    # the rounding of b and of the forward products through the solve (4: not
    # quite independent), and that of x itself
    bar = (grow * eps + store) * (1 + 4 * _amplified(nx, ny, xper, yper, cells)
                                  * np.linalg.norm(b) / np.linalg.norm(want))
    print(f"\n{nx}x{ny} {int(xper)}{int(yper)} {precision} cells={cells}: err {err:.1e} "
          f"bar {bar:.1e}")
    assert err <= bar
    w = np.random.default_rng(nx).standard_normal((ny, nx))
    c2v = not cells and not (xper and yper)
    if c2v:
        w = w.astype("f4").astype(float) if store else w
        q = np.pad(w, ((1, 0), (1, 0)), mode="constant")
        if xper:
            q[1:, 0] = w[:, -1]
        if yper:
            q[0, 1:] = w[-1]
        b = 0.25 * (q[:-1, :-1] + q[:-1, 1:] + q[1:, :-1] + q[1:, 1:]) * wet
    else:
        w = b = w * wet - (w.mean() if singular else 0.0)
    x = solve(w, c2v)
    r = _apply(x, xper, yper, cells, wet) - b
    if singular:
        r -= r.mean()
    res, bar = np.linalg.norm(r), 8 * np.linalg.norm(x) * (grow * eps + store) \
        + (grow * eps + store) * np.linalg.norm(b)
    print(f"  noise: residual {res:.1e} bar {bar:.1e}")
    assert res <= bar


@pytest.mark.parametrize("nx,ny,tile,xper", [(1100, 1030, 32, False), (4000, 2000, 64, True)])
def test_masked_writes(dev, nx, ny, tile, xper):
    """The capacitance solve around these tiles: the last pass writes at the
    unknowns only, no halo images of its own."""
    assert _tile(nx - 1, ny - 1) == tile

    def islands(msk):
        msk[ny // 3:ny // 3 + 9, nx // 4:nx // 4 + 14] = 0
        msk[ny // 2 + 40, nx // 2 + 7] = 0
    m, ps = _solver(nx, ny, xper, False, "fp64", False, islands)
    assert ps.method == "modal_capacitance"
    wet = (ps.msk[3:-3, 3:-3] != 0) * 1.0
    b = np.zeros((ny + 6, nx + 6))
    b[3:-3, 3:-3] = np.random.default_rng(3).standard_normal((ny, nx)) * wet
    x = torch.full(b.shape, 7.0, dtype=torch.float64, device=dev)
    ps.solve(T(b, dev), x)
    full = N(x)
    got = full[3:-3, 3:-3]
    assert np.all(got[wet == 0] == 7.0)
    filled = full.copy()
    m.mesh.fill(filled)
    assert np.array_equal(filled, full)
    got = got * wet
    res = np.linalg.norm(_apply(got, xper, False, False, wet) - b[3:-3, 3:-3])
    # two solves of that kind and the dense product between them
    bar = 3 * 8 * np.linalg.norm(got) * 8 * np.sqrt(max(nx, ny) / 2) * 2.0 ** -53
    print(f"\nmasked {nx}x{ny}: residual {res:.1e} bar {bar:.1e}")
    assert res <= bar

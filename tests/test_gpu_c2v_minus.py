"""centerstovertices less a vertex field in one kernel: bit for bit the two
operators one after the other, every entry of the padded array."""
import numpy as np
import pytest
import torch

from fluids2d_amd import Model, Param
from fluids2d_amd import operators as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("ny,nx,xper", [(8, 8, True), (17, 31, False), (64, 130, True)])
def test_c2v_minus(dev, ny, nx, xper, precision):
    p = Param()
    for k, v in dict(model="advection", nx=nx, ny=ny, xperiodic=xper, yperiodic=False,
                     precision=precision).items():
        setattr(p, k, v)
    m = Model(p).mesh
    dt = torch.float64 if precision == "fp64" else torch.float32
    rng = np.random.default_rng(nx)
    c, f, old = (torch.from_numpy(rng.standard_normal(m.shape)).to(dev, dt) for _ in range(3))
    c[5, 5] = float("nan")
    f[6, 7] = float("inf")
    want, got = old.clone(), old.clone()
    op.centerstovertices(m, c, want)
    op.addto_terms(want, [f], [-1.0])
    op.centerstovertices_minus(m, c, f, got)
    assert torch.equal(want.isnan(), got.isnan())
    assert torch.equal(want.nan_to_num(), got.nan_to_num())
    with pytest.raises(ValueError):
        op.centerstovertices_minus(m, c, f[1:], got)

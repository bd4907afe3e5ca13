"""The transport stage on sizes that the tile does not divide (whole tiles,
the last of a row or column of tiles moved back over its neighbour) and on
interiors smaller than a tile (bounds-tested tiles), bit for bit against the
oracle: every entry of the tendency and of the update, halo included."""
import pytest

import test_gpu_kernels as K
from test_gpu_kernels import L  # noqa: F401  (a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xper,yper,integ", [(False, False, "rk3"), (True, False, "enrk3"),
                                             (True, True, "rk3"), (False, True, "ef")])
@pytest.mark.parametrize("ny,nx,tile", [
    (17, 65, 0), (16, 127, 0), (31, 64, 0), (333, 501, 0), (9, 65, 1), (17, 33, 2),
    (33, 63, 3), (9, 129, 4),                            # moved tiles
    (15, 64, 0), (16, 63, 0), (8, 63, 1), (31, 33, 3)])  # smaller than a tile
def test_ragged(dev, L, xper, yper, integ, ny, nx, tile):  # noqa: F811
    K.test_transport_stage_bitexact(dev, L, xper, yper, "weno", integ, ny, nx, tile)

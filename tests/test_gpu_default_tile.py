"""The default tile at the lines of its rule: the last count of tiles that fits
the compute units at once, and the next (GPU: cffc_create needs a device)."""
import pytest

from cffc_amd import abi, euler2d
from cffc_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed,blocks,ni,nj,tile", [
    (False, (16, 16), 8, 8, (8, 8)),      # narrow blocks
    (False, (8, 8), 16, 16, (8, 8)),      # 256 tiles of 8 x 8: one a unit
    (False, (13, 5), 16, 16, (16, 8)),    # 260
    (False, (32, 20), 16, 16, (16, 8)),   # 1,280 of 16 x 8: five a unit
    (False, (641, 1), 16, 16, (16, 16)),
    (False, (32, 24), 16, 16, (16, 16)),  # 768 of 16 x 16: three a unit
    (False, (769, 1), 16, 16, (16, 8)),
    (False, (192, 1), 24, 32, (16, 16)),
    (False, (18, 12), 17, 17, (16, 8)),   # 1,296 of 16 x 8, but 864 of 16 x 16
    (False, (18, 12), 24, 24, (16, 8)),
    (False, (33, 1), 33, 33, (16, 8)),
    (False, (93, 1), 33, 33, (32, 16)),
    (True, (51, 5), 16, 8, (8, 8)),       # 255 of 16 x 8
    (True, (16, 16), 16, 8, (16, 8)),
    (True, (16, 4), 64, 64, (32, 16)),    # 512 of 32 x 16
    (True, (96, 1), 64, 64, (32, 16)),    # 768
    (True, (20, 5), 64, 64, (32, 16)),    # 800, half as many as of 32 x 8
    (True, (51, 1), 72, 72, (32, 16)),    # 765
    (True, (53, 1), 72, 72, (32, 8)),     # 795, more than half
    (True, (31, 3), 64, 36, (32, 8)),     # 558: three a unit, of 32 x 8 four
    (True, (29, 4), 64, 36, (32, 16)),    # 696: three a unit, of 32 x 8 five
    (True, (37, 9), 33, 33, (32, 8)),
])
def test_default_tile(mixed, blocks, ni, nj, tile):
    m = M.cartesian(blocks[0], blocks[1], ni, nj)
    m.set_wo_from_initial(M.riemann_4quadrant(m))
    g = euler2d.Euler2DQuadBlocks(m, abi.Scheme(flux_precision=abi.FLUX_FP32 if mixed else abi.FLUX_FP64))
    t = g.get_tile()
    g.close()
    assert tuple(t) == tile

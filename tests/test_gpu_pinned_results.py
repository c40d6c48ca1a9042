"""States read into memory that the runtime knows (pinned, or a device's) at
the size from which results into pageable memory go through pinned chunks, and
below it: the same bytes as into pageable memory."""
import ctypes

import numpy as np
import pytest
import torch

from cffc_amd import abi, euler2d
from cffc_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [4, 12])   # 2 and 19 MB
@pytest.mark.parametrize("where", ["pinned", "device"])
def test_result_in_known_memory(blocks, where):
    m = M.cartesian(blocks, blocks, 64, 64)
    W0 = M.density_perturbation(m, M.riemann_4quadrant(m), amplitude=0.01, seed=3)
    m.set_wo_from_initial(W0)
    g = euler2d.Euler2DQuadBlocks(m, abi.Scheme())
    g.set_W(W0)
    want = g.get_W()
    out = torch.zeros((g.ncell, 4), dtype=torch.float64, device="cuda" if where == "device" else "cpu",
                      pin_memory=where == "pinned")
    torch.cuda.synchronize()
    rc = euler2d.load().cffc_get_W(g.h, ctypes.cast(out.data_ptr(), ctypes.POINTER(ctypes.c_double)), g.ncell)
    g.close()
    assert rc == 0
    assert np.array_equal(out.cpu().numpy().view(np.uint64), np.asarray(want).reshape(-1, 4).view(np.uint64))

"""States through the chunked copies to host memory, below and above the size
where they begin and with a ragged last chunk; predictions of several batches
against one batch at a time.  Bit for bit."""
import numpy as np
import pytest

from cffc_amd import abi
from cffc_amd import mesh as M

pytestmark = pytest.mark.gpu


# 32 bytes a cell: just under 16 MiB, 16 MiB, a ragged 37 MB
@pytest.mark.parametrize("blocks", [(8, 8, 96, 85), (16, 16, 64, 32), (9, 7, 131, 143)])
def test_large_states_come_back(blocks):
    from cffc_amd import euler2d
    m = M.cartesian(*blocks)
    rng = np.random.default_rng(1)
    W0 = np.column_stack([rng.uniform(0.5, 2, m.ncell), rng.uniform(-1, 1, m.ncell), rng.uniform(-1, 1, m.ncell),
                          rng.uniform(0.5, 2, m.ncell)])
    g = euler2d.Euler2DQuadBlocks(m, abi.Scheme())
    for k in range(3):   # the buffers are used again
        g.set_W(W0 + k)
        np.testing.assert_array_equal(g.get_W(), W0 + k)
    g.close()


@pytest.mark.parametrize("count", [1, 4, 5, 8, 15])
def test_batches_of_predictions(count):
    from cffc_amd import unet
    net = unet.UNet(H=16, W=24, max_batch=4, seed=3)
    rng = np.random.default_rng(count)
    for l in range(net.nlayers):
        w, b = net.get_weights(l)
        net.set_weights(l, rng.normal(0, 0.1, w.shape), rng.normal(0, 0.1, b.shape))
    X = rng.normal(0, 1, (count, 16, 24, 8)).astype(np.float32)
    one = np.concatenate([net.predict(X[s:s + 1]) for s in range(count)])
    for _ in range(3):
        np.testing.assert_array_equal(net.predict(X), one)
    net.close()

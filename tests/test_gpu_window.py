"""Physical ghost states formed in the stage kernel's tile window: every
boundary type on every side, blocks whose last tile holds one column or row,
blocks smaller than a tile, and corner rules where a physical side meets a
neighbour.  FP64 against the CPU oracle (bitwise expected; the bound is the
parity tests' 1e-12), mixed against its own run through the exchange launch,
which a periodic side keeps."""
import numpy as np
import pytest

import oracle
from cffc_amd import abi
from cffc_amd import mesh as M

pytestmark = pytest.mark.gpu

F, R, E, C, P = (abi.BC_FIXED, abi.BC_REFLECTION, abi.BC_CONSTANT_EXTRAPOLATION, abi.BC_CHARACTERISTIC,
                 abi.BC_PERIODIC)
SIDES = [(F, E, R, R), (R, R, C, F), (C, C, E, R), (E, F, F, C), (R, C, R, E)]
BLOCKS = [(2, 2, 17, 9), (3, 1, 33, 17), (1, 2, 5, 3), (1, 1, 2, 2), (2, 1, 16, 16)]


def _case(sides, nbi, nbj, ni, nj):
    W, Ea, S, N = sides
    m = M.cartesian(nbi, nbj, ni, nj, bcs=dict(W=W, E=Ea, S=S, N=N), jitter=0.08, seed=ni + nj)
    W0 = M.density_perturbation(m, M.riemann_4quadrant(m), amplitude=0.05, seed=3)
    W0[:, 1] += 0.1
    m.set_wo_from_initial(W0)
    return m, W0


@pytest.mark.parametrize("blocks", BLOCKS)
@pytest.mark.parametrize("sides", SIDES)
def test_window_ghosts_match_the_oracle(sides, blocks):
    from cffc_amd import euler2d
    m, W0 = _case(sides, *blocks)
    o = oracle.Oracle(m, abi.Scheme())
    o.set_W(W0)
    rc, n, norms, _ = o.run(3)
    assert rc == 0 and n == 3
    Wo = o.get_W()
    for tile in (None, (16, 8), (32, 16), (8, 32)):
        g = euler2d.Euler2DQuadBlocks(m, abi.Scheme())
        if tile:
            g.set_tile(*tile)
        g.set_W(W0)
        rc, n, gn, _ = g.run_steps(3, graph=False)
        assert rc == 0 and n == 3
        W = g.get_W()
        assert np.max(np.abs(W - Wo) / np.maximum(np.abs(Wo), 1.0)) <= 1e-12
        assert np.allclose(gn, norms, rtol=1e-12, atol=0)
        g.close()


@pytest.mark.parametrize("sides", SIDES)
def test_mixed_window_ghosts_match_the_exchange_launch(sides):
    """The exchange launch serves a mesh with any periodic side: an unrelated
    periodic block in the same mesh keeps it for all blocks."""
    from cffc_amd import euler2d
    m, W0 = _case(sides, 2, 2, 17, 9)
    p, V0 = _case((P, P, P, P), 1, 1, 8, 8)
    both, _ = M.concat([m, p])
    # local time steps: the blocks of one case do not depend on the other's
    s = abi.Scheme(i_time_integration=abi.TIME_STEPPING_MULTISTAGE_OPTIMAL_SMOOTHING, n_stage=5, cfl_number=0.8,
                   local_time_stepping=abi.SCALAR_LOCAL_TIME_STEPPING, flux_precision=abi.FLUX_FP32)
    out = []
    for mesh, W in ((m, W0), (both, np.concatenate([W0, V0]))):
        g = euler2d.Euler2DQuadBlocks(mesh, s)
        g.set_tile(16, 8)
        g.set_W(W)
        rc, n, _, _ = g.run_steps(3)
        assert rc == 0 and n == 3
        out.append(g.get_W()[:m.ncell])
        g.close()
    assert np.array_equal(out[0], out[1])

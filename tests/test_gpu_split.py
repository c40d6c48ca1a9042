"""Split stage tiles (a thread per reconstructed variable, then per face)
against the unsplit ones, which tiles of 256 cells are: bit for bit, on blocks
that no tile divides, for every boundary type on every side, walls that reduce
the stencils, frozen limiters and resolution changes; and on both sides of the
number of tiles up to which a launch is split."""
import numpy as np
import pytest

from cffc_amd import abi
from cffc_amd import mesh as M

pytestmark = pytest.mark.gpu

F, R, E, C, P = (abi.BC_FIXED, abi.BC_REFLECTION, abi.BC_CONSTANT_EXTRAPOLATION, abi.BC_CHARACTERISTIC,
                 abi.BC_PERIODIC)
SIDES = [(F, E, R, R), (C, C, E, R), (E, F, F, C), (P, P, R, E)]
SPLIT = [(8, 8), (16, 4), (16, 8), (8, 16), (32, 4)]


def _case(sides, nbi, nbj, ni, nj):
    W, Ea, S, N = sides
    m = M.cartesian(nbi, nbj, ni, nj, bcs=dict(W=W, E=Ea, S=S, N=N), jitter=0.08, seed=ni + nj)
    W0 = M.density_perturbation(m, M.riemann_4quadrant(m), amplitude=0.05, seed=3)
    W0[:, 1] += 0.1
    m.set_wo_from_initial(W0)
    return m, W0


def _run(m, W0, tile, steps=4, steady_run=False):
    from cffc_amd import euler2d, steady
    g = euler2d.Euler2DQuadBlocks(m, steady.bump_scheme() if steady_run else abi.Scheme())
    g.set_tile(*tile)
    g.set_W(W0)
    if steady_run:
        g.set_parts([0, m.nblk])
        rc = g.run_steady(steps, 1e-12, 1e30)[0]   # frozen from the second step on
    else:
        rc = g.run_steps(steps, graph=False)[0]
    assert rc == 0
    W = g.get_W()
    g.close()
    return W


@pytest.mark.parametrize("blocks", [(2, 2, 17, 9), (3, 1, 33, 17), (1, 1, 2, 2), (2, 2, 24, 16)])
@pytest.mark.parametrize("sides", SIDES)
def test_split_tiles_give_the_same_bits(sides, blocks):
    m, W0 = _case(sides, *blocks)
    ref = _run(m, W0, (16, 16))
    for tile in SPLIT:
        np.testing.assert_array_equal(_run(m, W0, tile), ref)


def test_frozen_limiters():
    from cffc_amd import steady
    m, W0 = steady.bump_case(0.08, 0.5, nbi=3, nbj=2, ni=18, nj=10)
    ref = _run(m, W0, (16, 16), 12, True)
    for tile in SPLIT:
        np.testing.assert_array_equal(_run(m, W0, tile, 12, True), ref)


def test_resolution_changes():
    q = M.quadtree_box(nroot=4, n=8, max_level=1, refine=M.circle_refinement(0.3, band=0.0), jitter=0.1, seed=2)
    W0 = M.density_perturbation(q, M.cylindrical_explosion(q, radius=0.3), amplitude=0.01, seed=2)
    ref = _run(q, W0, (16, 16))
    for tile in SPLIT:
        np.testing.assert_array_equal(_run(q, W0, tile), ref)


@pytest.mark.parametrize("nb", [(32, 16), (27, 19)])
def test_the_last_split_launch_and_the_first_that_is_not(nb):
    """blocks of one 16 x 8 tile: 512 tiles are split, 513 are not"""
    m, W0 = _case(SIDES[0], nb[0], nb[1], 16, 8)
    np.testing.assert_array_equal(_run(m, W0, (16, 8), 2), _run(m, W0, (16, 16), 2))

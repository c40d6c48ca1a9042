"""The multigrid cycle's one-launch smoothing stages: tile windows that form
their own ghost cells (blocks no tile divides, many workgroups on the state
they update), first-order levels by cell list (connected blocks of more and of
fewer cells than one workgroup takes, disjoint meshes, blocks of 2 x 2 cells), every boundary
type on every side, repeated smoothings, and start-up on a coarse level that
keeps the full scheme.  Bitwise against the oracle."""
import numpy as np
import pytest

import oracle
from cffc_amd import abi
from cffc_amd import mesh as M
from cffc_amd import multigrid as MG
from cffc_amd import steady

pytestmark = pytest.mark.gpu

F, R, E, C = abi.BC_FIXED, abi.BC_REFLECTION, abi.BC_CONSTANT_EXTRAPOLATION, abi.BC_CHARACTERISTIC
SIDES = [(F, E, R, R), (C, F, E, R), (R, C, F, E), (E, R, C, F)]
# blocks, cells of one, levels: coarsest cells of a connected mesh in brackets
MESHES = [((1, 1, 8, 8), 3),      # [4] one block of 2 x 2
          ((3, 2, 40, 24), 3),    # [360] 10 x 6
          ((2, 1, 64, 64), 3),    # [512] 16 x 16: the largest in one workgroup
          ((2, 2, 64, 64), 3),    # [1024] listed, stage by stage
          ((3, 3, 44, 24), 2),    # [2376] 22 x 12
          ((2, 1, 72, 136), 3)]   # [1224] 18 x 34


def _part(sides, nbi, nbj, ni, nj):
    W, Ea, S, N = sides
    m = M.cartesian(nbi, nbj, ni, nj, bcs=dict(W=W, E=Ea, S=S, N=N), jitter=0.1, seed=ni + nj)
    Wf = M.freestream(0.4)
    m.wo[:] = Wf
    W0 = M.uniform_state(m, Wf)
    c = m.cell_centres()
    W0[:, 0] *= 1.0 + 0.1 * np.exp(-((c[:, 0] - 0.4) ** 2 + (c[:, 1] - 0.6) ** 2) / 0.03)
    return m, W0


def _run(parts, p, scheme, cycles=2, execute=False):
    m, _ = M.concat([q[0] for q in parts]) if len(parts) > 1 else (parts[0][0], None)
    W0 = np.concatenate([q[1] for q in parts])
    meshes = MG.hierarchy(m, p.levels)
    g = MG.FASMultigrid(m, scheme, p, meshes=meshes)
    o = oracle.OracleMG(meshes, scheme, p)
    for x in (g, o):
        x.set_W(W0)
        x.initialize()
    if execute:
        rg, ro = g.execute(cycles), o.execute(cycles)
        assert rg[0] == ro[0] == 0 and rg[1] == ro[1]
        np.testing.assert_allclose(rg[2], ro[2], rtol=1e-12, atol=0)
    else:
        for _ in range(cycles):
            assert g.cycle() == o.cycle() == 0
    for l in range(p.levels):
        np.testing.assert_array_equal(g.levels[l].get_U(), o.levels[l].get_U())
        np.testing.assert_array_equal(g.levels[l].get_W(), o.levels[l].get_W())
    g.close()


def _scheme(limiter=abi.LIMITER_VENKATAKRISHNAN):
    s = steady.bump_scheme(cfl=0.8)
    s.i_limiter = limiter
    return s


@pytest.mark.parametrize("mesh,levels", MESHES)
@pytest.mark.parametrize("sides", SIDES)
def test_levels_match_oracle(sides, mesh, levels):
    p = MG.MGParams(levels=levels, smooths_on_finest_level=2, smooths_on_coarsest_level=4)
    _run([_part(sides, *mesh)], p, _scheme())


@pytest.mark.parametrize("limiter", [abi.LIMITER_VENKATAKRISHNAN, abi.LIMITER_ZERO])
def test_disjoint_meshes_and_w_cycles(limiter):
    """with the zero limiter the finest level runs launch by launch"""
    p = MG.MGParams(levels=3, i_cycle=abi.MULTIGRID_W_CYCLE, pre_smooths=2, post_smooths=1)
    _run([_part(SIDES[0], *MESHES[1][0]), _part(SIDES[1], *MESHES[0][0]), _part(SIDES[2], 1, 2, 24, 40)], p,
         _scheme(limiter))


@pytest.mark.parametrize("first_order_coarse", [0, 1])
def test_start_up_on_the_coarsest_level(first_order_coarse):
    p = MG.MGParams(levels=3, fmg_cycles=3, first_order_coarse=first_order_coarse, smooths_on_coarsest_level=1)
    _run([_part(SIDES[1], *MESHES[1][0])], p, _scheme(), cycles=9, execute=True)

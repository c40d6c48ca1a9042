"""A multigrid solver whose settings change between two runs: execute replays
a recorded cycle, which has to be recorded again, so that it gives the same
states bit for bit as the launches themselves (set_graph(False)) in the same
sequence of calls."""
import numpy as np
import pytest

from cffc_amd import euler2d
from cffc_amd import mesh as M
from cffc_amd import multigrid as MG
from cffc_amd import serving, steady

pytestmark = pytest.mark.gpu


def _parts(g, m, starts, freeze):
    # tolerances that no case reaches
    g.set_parts(list(starts) + [m.nblk], np.full(len(starts), 1e-30), freeze)


SETTINGS = {
    # the second case frozen instead of the first, in newly allocated arrays
    "parts": lambda g, m, starts: _parts(g, m, starts, [0.0, 1e30]),
    "no parts": lambda g, m, starts: g.set_parts([0], []),
    "smoothing": lambda g, m, starts: g.set_residual_smoothing(0.6, 2),
    "tiles": lambda g, m, starts: [v.set_tile(*t) for v, t in zip(g.levels, [(16, 8), (8, 8), (4, 4)])],
    "limiters": lambda g, m, starts: g.levels[0].Freeze_Limiters(True),
}


@pytest.mark.parametrize("what", sorted(SETTINGS))
def test_setting_changed_between_runs(what):
    meshes = [serving.case_mesh(0.05, 0.4, 1), serving.case_mesh(0.08, 0.55, 1)]
    m, starts = M.concat([q[0] for q in meshes])
    W0 = np.concatenate([q[1] for q in meshes])
    out = []
    for graph in (True, False):
        g = MG.FASMultigrid(m, steady.bump_scheme(cfl=1.0), MG.MGParams(levels=3, absolute_tolerance=1e-30))
        g.set_graph(graph)
        g.set_W(W0)
        g.initialize()
        if what in ("parts", "no parts"):
            _parts(g, m, starts, [1e30, 0.0])   # the first case freezes at once
        rc, n, _ = g.execute(5, freeze_level=1.0 if "parts" in what else 0.0)
        assert (rc, n) == (0, 5)
        before = g.get_W()
        SETTINGS[what](g, m, starts)
        rc, n, _ = g.execute(5, freeze_level=1.0 if what == "parts" else 0.0)
        assert (rc, n) == (0, 5)
        out.append((before, g.get_W()))
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


def test_refused_parts_leave_no_parts():
    """After a cffc_mg_set_parts that is refused the solver has no parts: the
    next run is that of a solver that never had any, and there is no status."""
    meshes = [serving.case_mesh(0.05, 0.4, 1), serving.case_mesh(0.08, 0.55, 1)]
    m, starts = M.concat([q[0] for q in meshes])
    W0 = np.concatenate([q[1] for q in meshes])
    out = []
    for had_parts in (True, False):
        g = MG.FASMultigrid(m, steady.bump_scheme(cfl=1.0), MG.MGParams(levels=3, absolute_tolerance=1e-30))
        if had_parts:
            # both cases would stop at the third check
            g.set_parts(list(starts) + [m.nblk], np.full(len(starts), 1e30))
            with pytest.raises(euler2d.CffcError):
                g.set_parts(list(starts) + [m.nblk], np.full(len(starts), -1.0))
            with pytest.raises(euler2d.CffcError):
                g.part_status()
        g.set_W(W0)
        g.initialize()
        rc, n, _ = g.execute(6)
        assert (rc, n) == (0, 6)
        out.append(g.get_W())
        g.close()
    assert np.array_equal(out[0].view(np.uint64), out[1].view(np.uint64))

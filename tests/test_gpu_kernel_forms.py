"""The two forms of the tiled kernel against each other, bit for bit.

Steps without statistics, without a folded maximum, not at a caller's tau and with 256 cells a tile run a
kernel of their own (k_tile): long runs on large meshes.  All others run its general form, which the tests
with statistics and on small meshes reach.
"""
import numpy as np
import pytest

from radrhd_solver_amd import capi
from radrhd_solver_amd import mesh as M
from test_gpu_replays import PATHS, SEED, _solver

pytestmark = pytest.mark.gpu


def _run_kernel_forms(m, path, rad, runs):
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 100.0, 1.0])
    fields = M.init_radiation(m.n_cells, seed=SEED)
    out = {}
    for stats in (False, True):
        s = _solver(m, path, collect_stats=stats)
        assert s.step_form()["tile_cells"] == 256
        if rad:
            s.set_radiation(*fields)
        s.upload_W(W0)
        for n in runs:
            s.run(n)
        s.sync()
        st = s.stats()
        out[stats] = (*s.download(), s.face_flux(), st["steps"], st["t"], st["tau"], st["mlp_starts"], st["fix_calls"])
        assert (st["newton_iters"] > 0) == stats
        s.close()
    a, b = out[False], out[True]
    assert np.isfinite(b[0]).all()
    for k in range(3):
        assert np.array_equal(a[k], b[k])
    assert a[3:] == b[3:]
    assert path != "mixed_mlp" or a[6] > 0
    return a


@pytest.mark.parametrize("rad", [False, True])
@pytest.mark.parametrize("path", PATHS)
def test_plain_tile_kernel_equals_the_general_one(path, rad):
    """167,400 cells: 256 a tile on every path.  The first step of each run is the plain kernel's, the
    next ones fold; with statistics all are the general kernel's."""
    m = M.kuhn_box(31, 30, 30, seed=SEED)
    print("mesh", m.n_cells, m.n_faces, flush=True)
    _run_kernel_forms(m, path, rad, (1, 1, 1, 3, 1))


@pytest.mark.parametrize("path", ["fp64", "fp64_taub", "mixed", "mixed_taub", "mixed_mlp"])
def test_plain_tile_kernel_on_a_mesh_that_does_not_fold(path):
    """4,197,732 cells, 16,398 tiles: every step of a run is the plain kernel's, with the source."""
    m = M.kuhn_box(77, 77, 118, seed=SEED)
    print("mesh", m.n_cells, m.n_faces, flush=True)
    _run_kernel_forms(m, path, True, (5,))

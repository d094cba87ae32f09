"""rhllc_time_kernels times the step that rhllc_run takes."""
import numpy as np
import pytest

from radrhd_solver_amd import capi, surrogate
from radrhd_solver_amd import mesh as M

pytestmark = pytest.mark.gpu

SEED = 20261202


@pytest.mark.parametrize("schedule", [capi.SCHED_TILED, capi.SCHED_TWO_KERNEL])
@pytest.mark.parametrize("path", ["fp64", "mixed_mlp"])
@pytest.mark.parametrize("shape,folds", [((7, 6, 5), True), ((31, 30, 30), True), ((77, 77, 118), False)])
def test_the_timed_steps_are_those_of_a_run(shape, folds, path, schedule):
    """Twenty steps and the timed ones leave the state, the time and the counts that a run of as many
    leaves, also for the steps after them; a step that folds is one kernel, the others end with a dt kernel."""
    m = M.kuhn_box(*shape, seed=SEED)
    print("mesh", m.n_cells, flush=True)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 100.0, 1.0])
    out = []
    for timed in (True, False):
        kw = dict(precision=capi.PREC_MIXED, guess=capi.GUESS_MLP) if path == "mixed_mlp" else {}
        s = capi.Solver(m, cfl=0.4, schedule=schedule, **kw)
        if kw:
            s.set_mlp(surrogate.load(5 / 3))
        s.upload_W(W0)
        assert s.step_form()["folds"] == (folds and schedule == capi.SCHED_TILED)
        got = []
        for n in (5, 4):
            if timed:
                t = s.time_kernels(n)
                assert t["face_ms"] > 0 and t["step_ms"] >= t["face_ms"]
                if folds and schedule == capi.SCHED_TILED:
                    assert t["cell_ms"] == 0 and t["dt_ms"] == 0
                else:
                    assert t["dt_ms"] > 0
            else:
                s.run(20 + n)
            s.sync()
            st = s.stats()
            got.append((*s.download(), s.face_flux(), st["steps"], st["t"], st["tau"], st["max_speed"], st["mlp_starts"]))
            s.run(3)
        s.close()
        out.append(got)
    for a, b in zip(*out):
        assert all(np.array_equal(x, y) for x, y in zip(a[:3], b[:3])) and a[3:] == b[3:]

"""Graph replays against single launches, bit for bit.

rhllc_run captures a graph of 24 steps once its replays would serve 72 steps, so every run here that is
meant to replay is long enough and is checked to have replayed.  A graph holds its kernels' arguments by
value: a setter between two runs has to reach the second.
"""
import numpy as np
import pytest

import oracle as O
from radrhd_solver_amd import capi, surrogate
from radrhd_solver_amd import mesh as M
from rad_cases import physical_blast, table_path

pytestmark = pytest.mark.gpu

SEED = 20261202
PATHS = {
    "fp64": dict(),
    "fp64_previous": dict(guess=capi.GUESS_PREVIOUS),
    "fp64_taub": dict(eos=capi.EOS_TAUB),
    "mixed": dict(precision=capi.PREC_MIXED, guess=capi.GUESS_PREVIOUS),
    "mixed_taub": dict(precision=capi.PREC_MIXED, guess=capi.GUESS_PREVIOUS, eos=capi.EOS_TAUB),
    "mixed_mlp": dict(precision=capi.PREC_MIXED, guess=capi.GUESS_MLP),
}


def _solver(m, path, **kw):
    s = capi.Solver(m, cfl=0.4, **PATHS[path], **kw)
    if path == "mixed_mlp":
        s.set_mlp(surrogate.load(5 / 3))
    return s


def _fields(n):
    rng = np.random.default_rng(SEED)
    rad = M.init_radiation(n, seed=SEED)
    other = M.init_radiation(n, seed=SEED + 1)
    Tr = (np.eye(3) / 3 + 0.02 * rng.normal(size=(n, 3, 3))).astype(np.float32)
    return rad, other, Tr


def _stages(s, setters, W0, graph):
    """Each setter, then the state W0 and 73 or 97 steps from it (three or four graphs of 24, starting
    from either state buffer)."""
    got = []
    for k, (name, setter) in enumerate(setters):
        if W0 is not None:
            s.upload_W(W0)
        setter(s)
        before, steps = s.step_form()["replays"], (73, 97)[k % 2]
        s.run(steps, graph=graph)
        s.sync()
        assert s.step_form()["replays"] - before == (steps // 24 if graph else 0), name
        st = s.stats()
        got.append((name, *s.download(), st["steps"], st["t"], st["tau"], st["max_speed"], st["newton_iters"]))
    s.close()
    return got


def _compare(a, b):
    for x, y in zip(a, b):
        assert np.isfinite(y[1]).all(), y[0]
        assert np.array_equal(x[1], y[1]) and np.array_equal(x[2], y[2]) and x[3:] == y[3:], x[0]


@pytest.mark.parametrize("schedule", [capi.SCHED_TILED, capi.SCHED_TWO_KERNEL])
@pytest.mark.parametrize("path", PATHS)
def test_setters_between_replays(path, schedule):
    m = M.kuhn_box(8, 7, 6, seed=SEED)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 100.0, 1.0])
    rad, other, Tr = _fields(m.n_cells)
    weak = tuple(np.float32(1e-3) * a for a in rad[:2]) + tuple(rad[2:])
    model = surrogate.load(5 / 3).copy()
    model[: capi.MLP_PARAMS] *= np.float32(1.01)
    setters = [
        ("none", lambda s: None),
        ("none again", lambda s: None),
        ("radiation", lambda s: s.set_radiation(*weak)),
        ("opacities", lambda s: s.set_radiation(*weak[:2], *other[2:])),
        ("tensor", lambda s: s.set_radiation_tensor(Tr)),
        ("no tensor", lambda s: s.set_radiation_tensor(None)),
        ("statistics", lambda s: s.set_collect_stats(True)),
        ("no statistics", lambda s: s.set_collect_stats(False)),
        ("model", lambda s: s.set_mlp(model) if path == "mixed_mlp" else None),
        ("no radiation", lambda s: s.set_radiation(None, None)),
        ("time", lambda s: s.set_time(0.3 * m.h_min(), 7.0)),
    ]
    a, b = (_stages(_solver(m, path, schedule=schedule), setters, W0, graph) for graph in (True, False))
    _compare(a, b)
    for i, j in ((0, 2), (1, 3), (2, 4)):  # the setters matter
        assert not np.array_equal(a[i][2], a[j][2])


@pytest.mark.parametrize("path", PATHS)
def test_state_goes_on_over_replays(path):
    """Four runs one after the other, none from a fresh upload but the first."""
    m = M.kuhn_box(8, 7, 6, seed=SEED)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 100.0, 1.0])
    solvers = [_solver(m, path) for _ in range(2)]
    for s in solvers:
        s.upload_W(W0)
    _compare(*(_stages(s, [("none", lambda s: None)] * 4, None, graph) for s, graph in zip(solvers, (True, False))))


@pytest.mark.parametrize("path", ["fp64", "fp64_taub", "mixed"])
def test_tables_between_replays(path, tmp_path):
    """Opacity tables changed and removed between replays (physical states)."""
    m = M.kuhn_box(8, 7, 6, seed=SEED)
    W0, Ur, Fr = physical_blast(m, seed=5, ur_scale=1.0)
    hdr, data = M.read_table(table_path(tmp_path))
    setters = [
        ("table", lambda s: (s.set_opacity_table((hdr, data)), s.set_radiation(Ur, Fr))),
        ("the same", lambda s: None),
        ("another table", lambda s: s.set_opacity_table((hdr, data + 0.7))),
        ("no table", lambda s: (s.set_radiation(None, None), s.set_opacity_table(None))),
    ]
    a, b = (_stages(_solver(m, path), setters, W0, graph) for graph in (True, False))
    _compare(a, b)
    assert not np.array_equal(a[0][2], a[2][2]) and not np.array_equal(a[1][2], a[3][2])


@pytest.mark.parametrize("schedule", [capi.SCHED_TILED, capi.SCHED_TWO_KERNEL])
@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
def test_replays_of_the_periodic_shear_are_the_oracles_bits(eos, schedule):
    """FP64, 73 steps in three graphs and one single step."""
    m = M.kuhn_box(8, 7, 6, origin=(-0.5, -0.5, -0.5), periodic=7, seed=SEED)
    h = m.h_min()
    W0 = M.init_state(m, M.INIT_SHEAR, seed=SEED)
    st = O.State(m, W0, eos=eos)
    st.run(0.4, h, 73)
    s = capi.Solver(m, cfl=0.4, h_min=h, eos=eos, schedule=schedule)
    s.upload_W(W0)
    s.run(73)
    s.sync()
    assert s.step_form()["replays"] == 3
    W, U = s.download()
    for a, b in ((W, st.W), (U, st.U), (s.face_flux(), st.face_flux)):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
    s.close()


def test_graphs_are_captured_at_72_steps_worth():
    m = M.kuhn_box(5, 4, 3, seed=SEED)
    s = capi.Solver(m, cfl=0.4)
    s.upload_W(M.init_state(m, M.INIT_BLAST))
    for steps, replays in ((72, 0), (25, 1), (24, 0), (73, 3)):  # a run's first step is not in a graph
        before = s.step_form()["replays"]
        s.run(steps)
        assert s.step_form()["replays"] - before == replays, steps
    s.close()


def test_replays_on_a_mesh_that_does_not_fold():
    """The mixed step with the source and the surrogate start, 73 steps replayed and single."""
    m = M.kuhn_box(77, 77, 118, seed=SEED)
    print("mesh", m.n_cells, m.n_faces, flush=True)
    W0 = M.init_state(m, M.INIT_BLAST)
    fields = M.init_radiation(m.n_cells, seed=SEED)
    out = []
    for graph in (True, False):
        s = _solver(m, "mixed_mlp")
        s.set_radiation(*fields)
        s.upload_W(W0)
        s.run(73, graph=graph)
        s.sync()
        form = s.step_form()
        assert not form["folds"] and form["replays"] == (3 if graph else 0)
        st = s.stats()
        out.append((*s.download(), st["t"], st["tau"], st["mlp_starts"]))
        s.close()
    a, b = out
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2:] == b[2:]

"""The FP64 step's unscaled quotients and roots (ordinary states) against the oracle, bit for bit.

The line between them and the scaled ones is at 2^-100 and 2^100 for density, pressure and energy
and at 2^-300 for the momentum: flows scaled to both sides of each line, to the line itself, and
with single cells beyond it, so that a step's faces, its cells and both together take either form.
"""
import numpy as np
import pytest

import oracle as O
from radrhd_solver_amd import capi
from radrhd_solver_amd import mesh as M

pytestmark = pytest.mark.gpu

SEED = 20261202


def _check(W0, m, eos, steps=12):
    h = m.h_min()
    st = O.State(m, W0, eos=eos)
    st.run(0.4, h, steps)
    s = capi.Solver(m, cfl=0.4, h_min=h, eos=eos)
    s.upload_W(W0)
    s.run(steps)
    s.sync()
    W, U = s.download()
    for a, b in ((W, st.W), (U, st.U), (s.face_flux(), st.face_flux)):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
    s.close()


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
@pytest.mark.parametrize("log2", [-140, -101, -100, -99, -60, 0, 60, 88, 92, 99, 100, 140])
def test_scaled_flows(log2, eos):
    """A blast with rho and p scaled by 2^k: its lowest values lie on one side of the line and its
    highest on the other from k = -101 to -88 and from 88 to 99."""
    m = M.kuhn_box(7, 6, 5, seed=SEED)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 1000.0, 1.0])
    W0[:, [0, 4]] *= 2.0 ** log2
    _check(W0, m, eos)


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
@pytest.mark.parametrize("v", [0.0, 1e-30, 2.0 ** -299, 2.0 ** -301, 1e-160, 1e-300, 5e-324])
def test_tiny_velocities(v, eos):
    """Gas of one state but for a velocity of size v along x in half of the cells."""
    m = M.kuhn_box(6, 5, 4, seed=SEED)
    W0 = M.init_state(m, M.INIT_UNIFORM, params=[1.0, 0.0, 0.0, 0.0, 0.5])
    W0[::2, 1] = v
    _check(W0, m, eos, steps=4)


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
@pytest.mark.parametrize("cell", [(1e-35, 0.5), (1.0, 1e-33), (1e31, 2e31), (1.0, 1e-200)])
def test_single_cells_beyond_the_line(cell, eos):
    m = M.kuhn_box(8, 7, 6, seed=SEED)
    W0 = M.init_state(m, M.INIT_SHEAR)
    W0[7, 0], W0[7, 4] = cell
    W0[7, 1:4] = 0.0
    _check(W0, m, eos, steps=6)


def _check_starts(W0, m, eos, steps):
    """Each step's W from its U, cell by cell, with the scaled quotients and the stored pressure as
    the start.  Cells that PhysPressureFix rewrote are left out: they hold its pressure, 1e-12, and a U
    of its own.  Returns the share of the others."""
    s = capi.Solver(m, cfl=0.4, h_min=m.h_min(), eos=eos, guess=capi.GUESS_PREVIOUS)
    s.upload_W(W0)
    W, fixed = s.download()[0], 0
    for _ in range(steps):
        s.run(1)
        start = W[:, 4].copy()
        W, U = s.download()
        ref, code, _ = capi.eval_c2p(U, guess=start, eos=eos)
        ok = W[:, 4] != 1e-12
        fixed += (~ok).sum()
        assert (code[ok] == 0).all()
        assert np.array_equal(W[ok].view(np.uint64), ref[ok].view(np.uint64))
    assert fixed == s.stats()["fix_calls"]
    s.close()
    return 1 - fixed / (steps * m.n_cells)


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
@pytest.mark.parametrize("log2", [-140, -100, 0, 92, 99, 140])
def test_previous_pressure_starts(log2, eos):
    m = M.kuhn_box(7, 6, 5, seed=SEED)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 1000.0, 1.0])
    W0[:, [0, 4]] *= 2.0 ** log2
    assert _check_starts(W0, m, eos, steps=8) > 0.9


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
@pytest.mark.parametrize("log10", [-323, -312, -308, -305, -303, -200, -31, -28, 31])
def test_previous_pressure_starts_beyond_the_line(log10, eos):
    """Moving gas whose U is ordinary and whose pressures are far from the line (up to a decade
    above the given power of ten; cold enough, the first quotient is the start over a number near 1)."""
    m = M.kuhn_box(12, 11, 10, seed=SEED)
    rng = np.random.default_rng(SEED)
    W0 = M.init_state(m, M.INIT_UNIFORM, params=[1.0, 0.1, 0.2, -0.15, 1.0])
    W0[:, 4] = 10.0 ** log10 * 10 ** rng.uniform(0, 1, m.n_cells)
    assert _check_starts(W0, m, eos, steps=2) > 0.1


def test_an_upload_of_ordinary_states_returns_to_the_unscaled_form():
    """The mark of a state beyond the line lasts until the next upload, whichever chunk of an upload
    the state comes in, with W alone or W and U, and through graph replays."""
    m = M.kuhn_box(39, 39, 39, seed=SEED)  # 355,914 cells: two chunks of W, four of W and U
    n = m.n_cells
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 10.0, 1.0])
    _, U0 = O.p2c(W0)
    s = capi.Solver(m, cfl=0.4, h_min=m.h_min())
    s.upload_W(W0)
    assert s.step_form()["unscaled"]
    for cell in (0, n // 2, n - 1):
        for whole in (False, True):
            W1 = W0.copy()
            W1[cell, 4] = 1e-33
            _, U1 = O.p2c(W1)
            s.upload(W1, U1) if whole else s.upload_W(W1)
            assert not s.step_form()["unscaled"]
            s.run(1)
            assert not s.step_form()["unscaled"]
            s.upload(W0, U0) if whole else s.upload_W(W0)
            assert s.step_form()["unscaled"]
            s.run(1)
            assert s.step_form()["unscaled"]
    s.close()


def test_the_mark_under_replays():
    m = M.kuhn_box(6, 5, 4, seed=SEED)
    h = m.h_min()
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 10.0, 1.0])
    W1 = W0.copy()
    W1[7, 4] = 1e-33
    s = capi.Solver(m, cfl=0.4, h_min=h)
    for W in (W1, W0, W1, W0):
        st = O.State(m, W)
        st.run(0.4, h, 73)
        s.upload_W(W)
        before = s.step_form()
        assert before["unscaled"] == (W is W0)
        s.run(73)
        s.sync()
        after = s.step_form()
        assert after["replays"] == before["replays"] + 3 and after["unscaled"] == (W is W0)
        for a, b in zip(s.download(), (st.W, st.U)):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
    s.close()


def test_a_ghost_state_beyond_the_line_marks_every_upload():
    m = M.kuhn_box(5, 4, 3, seed=SEED)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 10.0, 1.0])
    for p, unscaled in ((0.1, True), (1e-40, False)):
        w = np.array([[0.1, 0.9, 0.0, 0.0, p]])
        _, u = O.p2c(w)
        s = capi.Solver(m, cfl=0.4, out_source=(w[0], u[0]))
        for _ in range(2):
            s.upload_W(W0)
            assert s.step_form()["unscaled"] == unscaled
            s.run(1)
            assert s.step_form()["unscaled"] == unscaled
        s.close()

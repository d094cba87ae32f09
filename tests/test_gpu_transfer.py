"""State, flux and field transfers of a handle (caller's records <-> device numbering).

The transfers go through two 8 MB pinned chunks in turn; 355,914 cells take several chunks of
each kind (40 and 80 bytes a cell, 40 a face, 24 a cell for the radiation fields) with a ragged
last one, 6 and 630 cells a part of one.  Everything is a copy, or the FP64 step and source of
the oracle, so every comparison is for equal bits.
"""
import time

import numpy as np
import pytest

import oracle as O
from radrhd_solver_amd import capi
from radrhd_solver_amd import mesh as M

pytestmark = pytest.mark.gpu

SEED = 20261202
SHAPES = [(1, 1, 1), (7, 5, 3), (39, 39, 39)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_MIXED])
def test_records_round_trip(shape, precision):
    m = M.kuhn_box(*shape, seed=SEED)
    n = m.n_cells
    rng = np.random.default_rng(SEED)
    W = np.column_stack([rng.uniform(0.5, 2, n), rng.uniform(-0.3, 0.3, (n, 3)), rng.uniform(0.5, 2, n)])
    _, U = O.p2c(W)
    s = capi.Solver(m, precision=precision,
                    guess=capi.GUESS_PREVIOUS if precision == capi.PREC_MIXED else capi.GUESS_REFERENCE)
    L = capi._lib()
    recs = rng.random((n, 17))  # elem_t: W at 0, U at 40, 56 more bytes
    recs[:, :5], recs[:, 5:10] = W, U
    capi.check(L.rhllc_upload_state(s.h, recs.ctypes.data, 136, 0, 40))
    out = np.full((n, 17), -7.0)
    capi.check(L.rhllc_download_state(s.h, out.ctypes.data, 136, -1, 40))
    assert np.array_equal(out[:, 5:10], U)
    assert (out[:, :5] == -7.0).all() and (out[:, 10:] == -7.0).all()
    capi.check(L.rhllc_download_state(s.h, out.ctypes.data, 136, 96, 0))  # W and U elsewhere in the record
    assert np.array_equal(out[:, :5], U) and (out[:, 10:12] == -7.0).all()
    W1, U1 = s.download()
    assert np.array_equal(U1, U) and np.array_equal(W1, out[:, 12:17])
    if precision == capi.PREC_FP64:
        assert np.array_equal(W1, W)
    else:  # W is recovered from U: the c2p of the stored states
        assert np.allclose(W1, W, rtol=1e-9, atol=1e-12)
    s.upload_W(W)
    assert np.array_equal(s.download()[1], U)
    s.close()


@pytest.mark.parametrize("shape", SHAPES)
def test_fields_and_fluxes_reach_their_cells_and_faces(shape):
    m = M.kuhn_box(*shape, seed=SEED)
    W0 = M.init_state(m, M.INIT_BLAST, params=[0.5, 0.5, 0.5, 0.3, 1.0, 100.0, 1.0])
    rad = M.init_radiation(m.n_cells, seed=SEED)
    h = m.h_min()
    st = O.State(m, W0)
    st.run_rad(0.4, h, 1, *rad)
    s = capi.Solver(m, cfl=0.4, h_min=h)
    s.set_radiation(*rad)
    s.upload_W(W0)
    s.run(1)
    s.sync()
    W, U = s.download()
    assert np.array_equal(W, st.W) and np.array_equal(U, st.U)
    assert np.array_equal(s.face_flux(), st.face_flux)
    s.close()


def test_a_download_of_neither_part_waits():
    """It copies nothing, but the steps before it are done when it returns, as with either part."""
    m = M.kuhn_box(48, 48, 48, seed=SEED)
    s = capi.Solver(m, cfl=0.4)
    s.upload_W(M.init_state(m, M.INIT_BLAST))
    L, out = capi._lib(), np.full((m.n_cells, 5), -7.0)

    def rest():  # seconds left for sync after the call, of a run of 2,000 steps
        s.run(2000)
        t0 = time.perf_counter()
        capi.check(L.rhllc_download_state(s.h, out.ctypes.data, 40, -1, -1))
        t1 = time.perf_counter()
        s.sync()
        return t1 - t0, time.perf_counter() - t1

    rest()
    waited, left = rest()
    print("waited", waited, "left", left)
    assert (out == -7.0).all() and left < 0.25 * (waited + left)
    s.close()

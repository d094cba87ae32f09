"""Mixed path: the cell record is the same whichever kernel forms it, and a tiled step's states are
its face fluxes' to the rounding of FP64 (the 1e-5 of a comparison with another schedule would let a
small fault of a tile size pass)."""
import numpy as np
import pytest

from radrhd_solver_amd import capi
from radrhd_solver_amd import mesh as M

pytestmark = pytest.mark.gpu

SEED = 20261202


def _table():  # one opacity at every density and temperature
    return np.array([-46.0, -23.0, 1.0, 9.0, 16.0, 1.0]), np.full((24, 8), -50.0)


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
def test_record_of_an_upload_is_the_record_of_a_step(eos):
    """A radiation source of tau = 0 leaves U as it is and forms the records anew from W recovered
    from U.  The W uploaded here are FP32 numbers, so W to 1e-9 gives the same FP32 values, and the
    step after it is that of the uploaded records bit for bit."""
    m = M.kuhn_box(9, 8, 7, origin=(-0.5, -0.5, -0.5), periodic=7, seed=SEED)
    W0 = M.init_state(m, M.INIT_SHEAR).astype(np.float32).astype(np.float64)
    out = []
    for source in (False, True):
        s = capi.Solver(m, cfl=0.4, precision=capi.PREC_MIXED, guess=capi.GUESS_PREVIOUS, eos=eos)
        s.upload_W(W0)
        U0 = s.download()[1]
        if source:
            s.set_opacity_table(_table())
            s.add_rad_flux(0.0, np.full(m.n_cells, 1e-12, np.float32), np.zeros((m.n_cells, 3), np.float32))
            assert np.array_equal(s.download()[1], U0)
        s.run(1)
        s.sync()
        out.append((s.download()[1], s.face_flux()))
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("eos", [capi.EOS_IDEAL, capi.EOS_TAUB])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 2, 2), (7, 5, 3), (16, 16, 16), (30, 30, 30), (31, 30, 30)])
def test_tiled_step_is_the_sum_of_its_face_fluxes(shape, eos):
    """Tiles of 64 and 256 cells, part of one, whole and ragged last ones.  The downloaded fluxes are
    formed face by face from the mesh's own cell pairs, the step's from the tile-local ones; U moves by
    tau / V times their signed sum.  A sum of four terms, its factor and the difference from U are each
    off by at most a few roundings of the largest term: 16 units of 2^-53 of their sum of sizes."""
    m = M.kuhn_box(*shape, seed=SEED)
    print("mesh", m.n_cells, m.n_faces, flush=True)
    rng = np.random.default_rng(SEED)
    n = m.n_cells
    W0 = np.column_stack([rng.uniform(0.5, 2, n), rng.uniform(-0.3, 0.3, (n, 3)), 10 ** rng.uniform(-1, 2, n)])
    tau = 0.4 * m.h_min()
    s = capi.Solver(m, cfl=0.4, precision=capi.PREC_MIXED, guess=capi.GUESS_PREVIOUS, eos=eos)
    s.upload_W(W0)
    U0 = s.download()[1]
    s.step(tau)
    U, F = s.download()[1], s.face_flux()
    s.close()
    sign = 2.0 * ((m.cells["sign_n"].astype(np.int64)[:, None] >> np.arange(4)) & 1) - 1.0
    terms = (tau / m.cells["V"])[:, None, None] * sign[:, :, None] * F[m.cells["id_faces"]]
    # the E flux is the sum of the fluxes of D and E - D, so its terms are bounded by both
    size = np.abs(U0) + np.abs(terms).sum(axis=1)
    size[:, 4] += size[:, 0]
    assert np.all(np.abs(U0 - terms.sum(axis=1) - U) <= 16 * 2.0 ** -53 * size)

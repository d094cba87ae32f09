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

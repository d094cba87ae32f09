"""Which meshes take tiles of 64 cells: on both sides of every line of the rule, in rounds of one
256-cell tile on each compute unit (FP64: up to 0.75, from 1 to 1.5 and from 2 to 2.25; mixed: up to 2.5)."""
import pytest

from radrhd_solver_amd import capi
from radrhd_solver_amd import mesh as M

pytestmark = pytest.mark.gpu

SEED = 20261202
# rounds -> FP64, mixed
EXPECT = {0.01: (64, 64), 0.74: (64, 64), 0.76: (256, 64), 0.99: (256, 64), 1.01: (64, 64), 1.49: (64, 64),
          1.51: (256, 64), 1.99: (256, 64), 2.01: (64, 64), 2.24: (64, 64), 2.26: (256, 64), 2.49: (256, 64),
          2.51: (256, 256), 3.1: (256, 256)}


@pytest.mark.parametrize("rounds", EXPECT)
def test_cells_per_tile(rounds):
    layer = capi.device_query(0)["cus"] * 256 / 6 / 100  # hexes of a round in each of 100 columns
    m = M.kuhn_box(10, 10, round(rounds * layer), seed=SEED)
    print("mesh", m.n_cells, flush=True)
    for k, kw in enumerate((dict(), dict(precision=capi.PREC_MIXED, guess=capi.GUESS_PREVIOUS))):
        s = capi.Solver(m, **kw)
        assert s.step_form()["tile_cells"] == EXPECT[rounds][k]
        s.close()


def test_two_kernel_step_has_no_tiles():
    s = capi.Solver(M.kuhn_box(3, 3, 3, seed=SEED), schedule=capi.SCHED_TWO_KERNEL)
    assert s.step_form()["tile_cells"] == 0
    s.close()

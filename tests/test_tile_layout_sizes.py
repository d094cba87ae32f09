"""The tiled step's host layout at both tile sizes that handles use (no GPU): the checks of
test_tile_layout at 64 and 256 cells a tile, with part of one tile, whole and ragged last tiles."""
import functools

import pytest

import test_tile_layout as layout
from radrhd_solver_amd import capi
from radrhd_solver_amd import mesh as M


@pytest.mark.parametrize("cells", [64, 256])
@pytest.mark.parametrize("reorder", [True, False])
@pytest.mark.parametrize("shape,kw", [((1, 1, 1), {}), ((2, 2, 2), {}), ((4, 4, 2), {}), ((5, 4, 3), {}),
                                      ((8, 8, 2), {}), ((12, 10, 9), {}), ((8, 8, 8), dict(periodic=7))])
def test_layout_matches_the_mesh_records(monkeypatch, cells, reorder, shape, kw):
    monkeypatch.setattr(layout, "T", cells)
    monkeypatch.setattr(capi, "tile_layout", functools.partial(capi.tile_layout, tile_cells=cells))
    m = M.kuhn_box(*shape, seed=5, **kw)
    L = layout._check(m, reorder)
    assert (L["tile_extra"].size > 0) == (m.n_cells > cells)


def test_other_tile_sizes_are_refused():
    m = M.kuhn_box(2, 2, 2, seed=5)
    for cells in (0, 63, 128, 512, -64):
        with pytest.raises(capi.RhllcError, match="64 or 256"):
            capi.tile_layout(m, tile_cells=cells)

"""Setting a context up: the tables that threads fill, and the meshes that are
refused."""
import numpy as np
import pytest

from adfvm_amd import _lib, context, meshgen
from tests import casefactory as cf
from tests import test_tiles
from tests.test_tiles import shim  # noqa: F401

THREADED = {
    'box': lambda: meshgen.permute_and_rcm(meshgen.periodic_box((41, 37, 45)), seed=3),
    'walls': lambda: meshgen.box((41, 37, 45)),
    'o_grid': lambda: meshgen.o_grid(301, 150),
}


@pytest.mark.parametrize('name', sorted(THREADED))
def test_tables_filled_by_threads(shim, name, monkeypatch):  # noqa: F811
    """45150 to 68265 cells: every table is filled by several threads."""
    monkeypatch.setitem(test_tiles.MESHES, name, THREADED[name])
    test_tiles.test_tile_tables(shim, name)


@pytest.mark.parametrize('cell', [0, 20000, -1])
def test_first_invalid_cell_is_reported(cell, monkeypatch):
    """A mesh is refused for its first invalid cell, whichever thread sees it;
    nothing of it has reached the device by then."""
    monkeypatch.setattr(context, '_need_torch', lambda: None)
    case = cf.CaseDef(meshgen.box((31, 30, 29)), {}, 1e-3)
    m = case.mesh
    m.cellFaces = m.cellFaces.copy()
    m.cellOwner = m.cellOwner.copy()
    m.cellFaces[cell, 3] = m.nFaces
    m.cellFaces[-1, 4], m.cellOwner[-1, 4] = m.nFaces - 1, 0
    with pytest.raises(_lib.LibraryError, match='cellFaces out of range'):
        case.context(np.float32)
    if cell == 0:
        m.cellFaces[0, 3] = 0
        with pytest.raises(_lib.LibraryError, match='boundary face in a neighbour slot'):
            case.context(np.float32)

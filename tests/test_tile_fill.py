"""Tiles of walls meshed finer along one axis stay compact: at most a tenth more of them than full
tiles would be (a tile is halved when its block rows have too many columns), each node in one."""
import numpy as np
import pytest

from cvfes_amd import _lib
from cvfes_amd.mesh import tube_geometry
from tests.test_gpu_tiles import tile_rows


@pytest.mark.parametrize("nt,nz,length", [(300, 40, 3.0), (64, 400, 3.0), (160, 120, 12.0), (96, 90, 0.4)])
def test_tiles_are_nearly_full(nt, nz, length):
    if not _lib.LIB_PATH.exists():
        pytest.skip("libcvfes_mi355x.so not built")
    nodes, el, _ = tube_geometry(nt, nz, 0.3, length)
    rows, _, _ = tile_rows(nodes, el)
    assert np.array_equal(np.sort(rows[rows >= 0]), np.arange(nodes.shape[0]))
    assert len(rows) <= 1.1 * np.ceil(nodes.shape[0] / _lib.TILE_ROWS)

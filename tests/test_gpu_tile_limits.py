"""3D Joseph tiles that fill the LDS are taken, and give the default tile's bits."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu


# slots a row as they are and padded to an odd number, bytes: 22, 61952 and 23, 64768 (past 64 KB with the
# pose tables); 30, 61440 and 31, 63488; 32, 159744 and 33, 164736 (past a workgroup's 160 KB)
@pytest.mark.parametrize("tile", [(16, 20, 20), (8, 28, 30), (16, 30, 37)], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_tiles_that_fill_the_lds(tile, dtype):
    import elsa_amd as E

    g = oracle.circle_geometry(3, (37, 45, 50), 15, 360, 400.0, 100.0, det=(80, 60))
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(2).standard_normal(g.sino_shape).astype(dtype)
    ref = op.applyAdjoint(y)
    op.tile(*tile)
    np.testing.assert_array_equal(op.applyAdjoint(y), ref)

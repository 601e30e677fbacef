"""Back projections of two driving axes in a launch each (few poses over a large volume): against the oracle, with the
same bits whatever the tile, alone and in a batch with a small problem."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu

# volumes of a million voxels, 5 poses of few rays: a launch for each axis' tiles
CASES = {3: ((105, 90, 112), (60, 50)), 2: ((1200, 900), (700,))}


def _geometry(dim):
    vol, det = CASES[dim]
    n = max(vol)
    return oracle.circle_geometry(dim, vol, 5, 360, 4.0 * n, 1.0 * n, det=det,
                                  angles_deg=np.array([0.0, 100.0, 45.0, 200.0, 271.0], np.float32))


@pytest.mark.parametrize("dim,method,dtype", [(3, "joseph", np.float32), (3, "joseph", np.float64),
                                              (3, "siddon", np.float32), (2, "siddon", np.float64)], ids=str)
def test_back_projection_of_few_poses(dim, method, dtype):
    import elsa_amd as E

    g = _geometry(dim)
    cls = E.JosephsMethodCUDA if method == "joseph" else E.SiddonsMethodCUDA
    op = cls(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(3).random(g.sino_shape).astype(dtype)
    got = op.applyAdjoint(y)
    f32 = dtype == np.float32
    if method == "joseph":
        mode = oracle.MODE_EXACT_WEIGHTS if f32 else oracle.MODE_DIRECT
        ref = oracle.joseph(g, y.astype(np.float64), adjoint=True, mode=mode, acc64=True)
        # positive terms: the product, an axis' sum and the voxel are rounded, and each term to half a unit (2^-50: max |y|
        # is below 1 and the slot bound 4096 for rays this far apart), for at most 200 rays a voxel
        eps = 2.0 ** -24 if f32 else 2.0 ** -52
        assert np.all(np.abs(got - ref) <= 3 * eps * ref * (1 + 1e-6) + 200 * 2.0 ** -51)
    else:
        # the lengths are the one-thread-per-ray kernel's, added in another order
        ref = cls(*geom_to_descriptors(g), dtype=dtype, kernels="simple").applyAdjoint(y)
        eps = 2.0 ** -24 if f32 else 2.0 ** -52
        assert np.all(np.abs(got - ref) <= 200 * eps * np.maximum(ref, 1.0))
    small = oracle.circle_geometry(dim, (9, 7, 8)[:dim], 4, 360, 90.0, 30.0, det=(12, 10)[:dim - 1])
    if f32:
        ops = [op, cls(*geom_to_descriptors(small), dtype=dtype)]
        ys = [y, np.random.default_rng(4).random(small.sino_shape).astype(dtype)]
        batch = E.ProjectorBatch(ops)
        assert batch.fused
        out = batch.unpack(batch.applyAdjoint(batch.pack(ys, adjoint_space=True)))
        np.testing.assert_array_equal(out[0].cpu().numpy(), got)
        np.testing.assert_array_equal(out[1].cpu().numpy(), ops[1].applyAdjoint(ys[1]))
    op.tile(5, 12, 12)
    np.testing.assert_array_equal(op.applyAdjoint(y), got)

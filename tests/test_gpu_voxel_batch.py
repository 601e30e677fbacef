"""Batches of 3D voxel projectors whose footprints differ in width: each operator's own bits, by columns (the
widest one's kernel for all) and with an operator that has none (the general kernel for all)."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu

# basis function and detector distance over source distance: 4, 5, 5 and 8 columns, none
OPS = {"bspline": ("BSplineVoxelProjectorCUDA", 0.05), "blob": ("BlobVoxelProjectorCUDA", 0.05),
       "pcblob": ("PhaseContrastBlobVoxelProjectorCUDA", 0.05), "blob8": ("BlobVoxelProjectorCUDA", 0.8),
       "wide": ("BlobVoxelProjectorCUDA", 2.0)}
SIZES = [((33, 28, 35), (50, 37), 12), ((9, 14, 6), (21, 30), 40), ((20, 20, 20), (64, 17), 5)]


@pytest.mark.parametrize("names", [("blob", "bspline"), ("bspline", "pcblob", "blob8"), ("blob8", "bspline", "blob"),
                                   ("bspline", "wide", "blob")], ids="-".join)
@pytest.mark.parametrize("tile", [None, (40, 8, 1)], ids=str)
def test_batch_of_mixed_widths(names, tile):
    import elsa_amd as E

    ops, xs, ys = [], [], []
    rng = np.random.default_rng(6)
    for name, (vol, det, poses) in zip(names, SIZES):
        cls, ratio = OPS[name]
        n = max(vol)
        g = oracle.circle_geometry(3, vol, poses, 360, 40.0 * n, 40.0 * n * ratio, det=det)
        ops.append(getattr(E, cls)(*geom_to_descriptors(g), dtype=np.float32))
        xs.append(rng.standard_normal(g.vol_shape).astype(np.float32))
        ys.append(rng.standard_normal(g.sino_shape).astype(np.float32))
    ref = [(op.apply(x), op.applyAdjoint(y)) for op, x, y in zip(ops, xs, ys)]
    if tile:
        for op in ops:
            op.tile(*tile)
    batch = E.ProjectorBatch(ops)
    assert batch.fused
    fwd = batch.unpack(batch.apply(batch.pack(xs)), adjoint_space=True)
    adj = batch.unpack(batch.applyAdjoint(batch.pack(ys, adjoint_space=True)))
    for f, a, (rf, ra) in zip(fwd, adj, ref):
        np.testing.assert_array_equal(f.cpu().numpy(), rf)
        np.testing.assert_array_equal(a.cpu().numpy(), ra)

"""The 3D voxel gather of footprints too wide for columns, where a wavefront takes several of a sum's parts: against
the oracle and, in a batch, each operator's own bits."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu

# volume, poses, detector distance over source distance (footprints of 13 and 29 pixels at most): eight parts in a
# wavefront each, four in one, eight in two, sixteen in four (and lanes without a voxel in the last block)
CASES = {"apart": ((40, 40, 40), 64, 2.0), "one": ((48, 51, 47), 33, 6.0), "two": ((37, 41, 36), 64, 6.0),
         "four": ((31, 29, 33), 130, 6.0)}


def _geometry(name):
    vol, poses, ratio = CASES[name]
    n = max(vol)
    return oracle.circle_geometry(3, vol, poses, 360, 40.0 * n, 40.0 * n * ratio, det=(50, 21))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["Blob", "PhaseContrastBlob"])
@pytest.mark.parametrize("name", list(CASES))
def test_wide_footprints(name, kind, dtype):
    import torch

    import elsa_amd as E

    g = _geometry(name)
    cls = getattr(E, kind + "VoxelProjectorCUDA")
    # positive pixels: the sums of the phase-contrast weights cancel, so both are held to the sum of magnitudes
    y = torch.from_numpy(np.random.default_rng(4).random(g.sino_shape).astype(np.float32))
    y = y.to(getattr(torch, dtype)).cuda()
    got = cls(*geom_to_descriptors(g), dtype=dtype).applyAdjoint(y).double().cpu().numpy()
    ref = cls(*geom_to_descriptors(g), dtype=np.float64).applyAdjoint(y.double()).cpu().numpy()
    mag = E.BlobVoxelProjectorCUDA(*geom_to_descriptors(g), dtype=np.float64).applyAdjoint(y.double()).cpu().numpy()
    # FP32: up to 1e5 sequential additions in parts of 1e4 (each half an ulp of its partial sum, random signs: 1e2 ulps)
    # and weights from distances known to 1e-6 of a radius; bfloat16 rounds the voxel
    eps = 2e-5 if dtype == "float32" else 2e-5 + 2.0 ** -8
    assert np.all(np.abs(got - ref) <= eps * (2.0 * mag.max() if kind != "Blob" else mag.max()))


def test_batch_of_wide_footprints():
    import elsa_amd as E

    rng = np.random.default_rng(5)
    ops, ys = [], []
    for name in CASES:
        g = _geometry(name)
        ops.append(E.BlobVoxelProjectorCUDA(*geom_to_descriptors(g), dtype=np.float32))
        ys.append(rng.standard_normal(g.sino_shape).astype(np.float32))
    batch = E.ProjectorBatch(ops)
    assert batch.fused
    for got, op, y in zip(batch.unpack(batch.applyAdjoint(batch.pack(ys, adjoint_space=True))), ops, ys):
        np.testing.assert_array_equal(got.cpu().numpy(), op.applyAdjoint(y))

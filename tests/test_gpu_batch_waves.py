"""3D Joseph forwards of small and large volumes in one batch, whose blocks take wavefronts of different shapes:
each operator's own bits, on detectors that leave remainders of either shape."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("det", [(1, 1), (33, 9), (64, 4), (65, 5), (130, 3), (257, 8)], ids=str)
def test_wavefronts_of_two_shapes(det):
    import elsa_amd as E

    rng = np.random.default_rng(3)
    ops, xs = [], []
    for vol, poses in (((17, 40, 33), 6), ((112, 5, 9), 5), ((111, 6, 20), 3), ((6, 7, 130), 4)):
        g = oracle.circle_geometry(3, vol, poses, 360, 3.0 * max(vol), 1.5 * max(vol), det=det)
        ops.append(E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=np.float32))
        xs.append(rng.standard_normal(g.vol_shape).astype(np.float32))
    batch = E.ProjectorBatch(ops)
    assert batch.fused
    for got, op, x in zip(batch.unpack(batch.apply(batch.pack(xs)), adjoint_space=True), ops, xs):
        np.testing.assert_array_equal(got.cpu().numpy(), op.apply(x))

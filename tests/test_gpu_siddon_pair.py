"""The Siddon back projection's launches against the oracle: rays of one driving axis, of two (both axes'
tiles in one launch) and of three, in both types, alone and in batches; tiles of every shape with the
same bits."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu

# vol, det, source and detector distance, angles: the axes that drive rays
CASES = {
    "2d": ((33, 20), (60,), 400.0, 100.0, tuple(range(0, 360, 9))),
    "2d_one": ((9, 33), (40,), 400.0, 100.0, (0.0, 5.0, -7.0)),
    "one": ((9, 33, 12), (20, 40), 400.0, 100.0, (0.0, 5.0, -7.0)),
    "two": ((17, 35, 40), (70, 50), 400.0, 100.0, tuple(range(0, 360, 24))),
    "three": ((10, 50, 9), (30, 120), 16.0, 8.0, (0.0, 40.0, 90.0, 200.0)),
}


def _geometry(name):
    vol, det, s2c, c2d, angles = CASES[name]
    return oracle.circle_geometry(len(vol), vol, len(angles), 360, s2c, c2d, det=det,
                                  angles_deg=np.asarray(angles, np.float32))


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("name", list(CASES))
def test_back_projection(name, dtype):
    import elsa_amd as E

    g = _geometry(name)
    op = E.SiddonsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(8).random(g.sino_shape).astype(dtype)
    got = op.applyAdjoint(y)
    # lengths are FP32 in both; the oracle sums one ray after another in the data's type, a few hundred terms
    # a voxel; positive data
    ref = oracle.siddon(g, y.astype(np.float64), adjoint=True)
    assert np.linalg.norm(got - ref) <= 5e-5 * np.linalg.norm(ref)
    tiles = ((4, 16), (7, 3), (1, 1), (16, 40)) if g.dim == 2 else ((8, 16, 16), (8, 22, 22), (1, 1, 1), (3, 6, 5),
                                                                     (16, 8, 9))
    for tile in tiles:
        op.tile(*tile)
        np.testing.assert_array_equal(op.applyAdjoint(y), got, err_msg=str(tile))
    y.reshape(-1)[3] = np.nan
    assert np.isnan(op.applyAdjoint(y)).all()


@pytest.mark.parametrize("names", [("two", "one"), ("two", "three"), ("one", "one"), ("2d", "2d_one")])
def test_batch_equals_each_operator(names):
    import elsa_amd as E

    gs = [_geometry(n) for n in names]
    ops = [E.SiddonsMethodCUDA(*geom_to_descriptors(g), dtype=np.float32) for g in gs]
    rng = np.random.default_rng(9)
    ys = [rng.standard_normal(g.sino_shape).astype(np.float32) for g in gs]
    batch = E.ProjectorBatch(ops)
    assert batch.fused
    out = batch.unpack(batch.applyAdjoint(batch.pack(ys, adjoint_space=True)))
    for got, op, y in zip(out, ops, ys):
        np.testing.assert_array_equal(got.cpu().numpy(), op.applyAdjoint(y))

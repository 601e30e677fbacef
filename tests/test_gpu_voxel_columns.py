"""The 3D voxel projectors by columns against the oracle: footprints of every column count that has a
kernel of its own and wider ones (the general kernels), volumes and detectors of odd sizes, footprints
that leave the detector, tiles of every shape with the same bits, alone and in a batch."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu

# basis function, detector distance over source distance: 4 (B-spline) and 5, 6, 8, 9, 13 columns
CASES = [("bspline", 0.05), ("blob", 0.05), ("blob", 0.35), ("bspline", 1.2), ("blob", 0.8), ("blob", 1.2),
         ("blob", 2.0)]
# (with 150 and 40 poses the gather sums in sixteen and four parts)
SIZES = [((13, 9, 11), (23, 17), 7), ((1, 1, 3), (5, 4), 150), ((33, 40, 7), (41, 3), 40)]


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _setup(kind, ratio, size, dtype):
    import elsa_amd as E

    vol, det, poses = size
    n = max(vol)
    angles = np.linspace(0.0, 300.0, poses).astype(np.float32)
    g = oracle.circle_geometry(3, vol, poses, 360, 20.0 * n, ratio * 20.0 * n, det=det, angles_deg=angles)
    if kind == "blob":
        return g, E.BlobVoxelProjectorCUDA, oracle.blob_lut(2.0, 10.83, 2, 100, dtype), 2.0
    return g, E.BSplineVoxelProjectorCUDA, oracle.bspline_lut(3, 2, 100, dtype), 1.5


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s[0])))
@pytest.mark.parametrize("kind,ratio", CASES)
def test_voxel_columns(kind, ratio, size, dtype):
    g, cls, lut, sup = _setup(kind, ratio, size, dtype)
    op = cls(*geom_to_descriptors(g), dtype=dtype)
    rng = np.random.default_rng(4)
    x = rng.random(g.vol_shape).astype(dtype)
    y = rng.random(g.sino_shape).astype(dtype)
    # FP32 rounds the distances, the weight and the result of positive terms, a few ulp each; FP64 only
    # sums in another order
    bar = 1e-6 if dtype == np.float32 else 1e-13
    got = op.apply(x)
    assert rel_l2(got, oracle.voxel(g, x, lut, sup, acc64=True)) <= bar
    assert rel_l2(op.applyAdjoint(y), oracle.voxel(g, y, lut, sup, adjoint=True, acc64=True)) <= bar
    for tile in ((32, 32), (7, 3), (1, 1), (200, 8), (16, 64)):
        op.tile(*tile, 1)
        np.testing.assert_array_equal(op.apply(x), got, err_msg=str(tile))
    x.reshape(-1)[1] = np.inf
    assert np.isnan(op.apply(x)).all()
    # an infinite pixel reaches the voxels whose footprints hold it and no others
    y[:] = 0
    y.reshape(-1)[y.size // 2] = 1
    held = op.applyAdjoint(y) != 0
    y.reshape(-1)[y.size // 2] = np.inf
    got = op.applyAdjoint(y)
    near = oracle.voxel(g, y, lut, 1.01 * sup, adjoint=True, acc64=True)
    assert not np.isfinite(got[held]).any() and np.isfinite(got[np.isfinite(near)]).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("spacing", [(0.5, 0.5, 0.5), (0.6, 0.6, 0.6), (1.5, 1.5, 1.5), (2.0, 0.8, 1.0)], ids=str)
@pytest.mark.parametrize("kind", ["blob", "bspline"])
def test_voxel_spacing(kind, spacing, dtype):
    """Footprints scale with the extrinsic matrix, which holds the voxel spacing: twice as wide (the
    general kernels) or wider, narrower and anisotropic (other column counts and tables)."""
    import elsa_amd as E

    vol, det = (17, 12, 21), (50, 44)
    poses = [oracle.geometry_pose(3, 300.0, 30.0, vol, det, angle_rad=a, vol_spacing=spacing)
             for a in (0.0, 0.4, 1.1, 1.6, 3.0)]
    g = oracle.geom_from_poses(3, vol, det, poses)
    cls = E.BlobVoxelProjectorCUDA if kind == "blob" else E.BSplineVoxelProjectorCUDA
    lut, sup = (oracle.blob_lut(2.0, 10.83, 2, 100, dtype), 2.0) if kind == "blob" else (
        oracle.bspline_lut(3, 2, 100, dtype), 1.5)
    op = cls(*geom_to_descriptors(g), dtype=dtype)
    rng = np.random.default_rng(8)
    x = rng.random(g.vol_shape).astype(dtype)
    y = rng.random(g.sino_shape).astype(dtype)
    bar = 1e-6 if dtype == np.float32 else 1e-13
    assert rel_l2(op.applyAdjoint(y), oracle.voxel(g, y, lut, sup, adjoint=True, acc64=True)) <= bar
    assert rel_l2(op.apply(x), oracle.voxel(g, x, lut, sup, acc64=True)) <= bar


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("vol,det,poses", [((1, 5), 9, 7), ((31, 17), 40, 33), ((24, 40), 61, 140)])
def test_gather_parts_2d(vol, det, poses, dtype):
    import elsa_amd as E

    g = oracle.circle_geometry(2, vol, poses, 360, 200.0, 60.0, det=(det,))
    op = E.BlobVoxelProjectorCUDA(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(6).random(g.sino_shape).astype(dtype)
    ref = oracle.voxel(g, y, oracle.blob_lut(2.0, 10.83, 2, 100, dtype), 2.0, adjoint=True, acc64=True)
    assert rel_l2(op.applyAdjoint(y), ref) <= (1e-6 if dtype == np.float32 else 1e-13)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("vol,det,poses", [((1, 5), 9, 7), ((31, 17), 40, 33), ((50, 60), 300, 1100)])
def test_forward_tiles_2d(vol, det, poses, dtype):
    """Tiles by the launch's size: narrow ones for few poses, up to 256 pixels for many."""
    import elsa_amd as E

    g = oracle.circle_geometry(2, vol, poses, 360, 200.0, 60.0, det=(det,))
    op = E.BlobVoxelProjectorCUDA(*geom_to_descriptors(g), dtype=dtype)
    x = np.random.default_rng(7).random(g.vol_shape).astype(dtype)
    got = op.apply(x)
    ref = oracle.voxel(g, x, oracle.blob_lut(2.0, 10.83, 2, 100, dtype), 2.0, acc64=True)
    assert rel_l2(got, ref) <= (1e-6 if dtype == np.float32 else 1e-13)
    for tile in (1, 16, 37, 256, 512):
        op.tile(tile, 1, 1)
        np.testing.assert_array_equal(op.apply(x), got, err_msg=str(tile))


@pytest.mark.parametrize("second", [("blob", 0.1), ("blob", 0.35), ("bspline", 1.2)])
def test_batch_of_columns(second):
    """Operators of one column count share the kernel by columns, others the general one."""
    import elsa_amd as E

    ops, xs, ys = [], [], []
    rng = np.random.default_rng(5)
    for (kind, ratio), size in zip([("blob", 0.05), second], SIZES[::2]):
        g, cls, _, _ = _setup(kind, ratio, size, np.float32)
        ops.append(cls(*geom_to_descriptors(g), dtype=np.float32))
        xs.append(rng.random(g.vol_shape).astype(np.float32))
        ys.append(rng.random(g.sino_shape).astype(np.float32))
    batch = E.ProjectorBatch(ops)
    assert batch.fused
    for got, op, x in zip(batch.unpack(batch.apply(batch.pack(xs)), adjoint_space=True), ops, xs):
        np.testing.assert_array_equal(got.cpu().numpy(), op.apply(x))
    for got, op, y in zip(batch.unpack(batch.applyAdjoint(batch.pack(ys, adjoint_space=True))), ops, ys):
        np.testing.assert_array_equal(got.cpu().numpy(), op.applyAdjoint(y))

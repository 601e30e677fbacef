"""Tiled Joseph back projections against the oracle with bars from the fixed-point unit itself: unit 2^(eg - 62), 2^eg the
power of two above max |y| times the slot bound, half a unit for each term that a voxel gets. The launches of three
driving axes in FP64, and the scale that every tile of a small 2D problem finds for itself."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu


def slot_bound(g):
    """Upper bound of the sum of |length x weight| that a slot can get: at most (2 / h + 2)^(dim - 1) rays a pose,
    h half the least distance of neighbouring rays at the volume."""
    dim, det = g.dim, g.det
    theta, dmin = 1e300, 1e300
    for p in range(g.nviews):
        pinv = np.asarray(g.Pinv[p], np.float64).ravel()
        m = np.array([[pinv[i + j * (dim + 1)] for j in range(dim)] for i in range(dim)])

        def direction(*uv):
            n = m @ np.array([*uv, 1.0])
            return n / np.linalg.norm(n)

        ends = [(0.5, n - 0.5, n / 2) for n in det[:dim - 1]]
        for uv in np.stack(np.meshgrid(*ends), -1).reshape(-1, dim - 1):
            for k in range(dim - 1):
                step = np.eye(dim - 1)[k]
                theta = min(theta, np.linalg.norm(direction(*(uv + step)) - direction(*uv)))
        c = np.asarray(g.C[p], np.float64)[:dim]
        dmin = min(dmin, np.linalg.norm(np.maximum(np.maximum(-c, c - np.asarray(g.vol)), 0.0)))
    h = 0.5 * theta * dmin
    return max(4096.0, g.nviews * (2.0 / h + 2.0) ** (dim - 1) * (1.7320509 if dim == 3 else 1.4142137))


def terms(g):
    """At most how many rays give a voxel a term: those through the box of two voxels a side around its centre,
    counted as the pixels of its projection's bounding rectangle."""
    dim, vol = g.dim, g.vol
    centre = np.stack(np.meshgrid(*[np.arange(n) + 0.5 for n in vol], indexing="ij"), -1).reshape(-1, dim)
    corners = np.stack(np.meshgrid(*[(-1.0, 1.0)] * dim), -1).reshape(-1, dim)
    count = np.zeros(len(centre))
    for p in range(g.nviews):
        P = np.asarray(g.P[p], np.float64).ravel().reshape(dim + 1, dim).T
        x = centre[:, None, :] + corners[None]
        q = x @ P[:, :dim].T + P[:, dim]
        uv = q[..., :dim - 1] / q[..., dim - 1:]
        n = np.ones(len(centre))
        for k in range(dim - 1):
            lo, hi = uv[..., k].min(1) - 1.0, uv[..., k].max(1) + 1.0
            n *= np.clip(np.minimum(hi, g.det[k]) - np.maximum(lo, 0.0) + 1.0, 0.0, None)
        count += n
    return count.reshape(vol).T


def check(got, g, y, mode, eps):
    ref = oracle.joseph(g, y, adjoint=True, mode=mode, acc64=True)
    mag = oracle.joseph(g, np.abs(y), adjoint=True, mode=mode, acc64=True)
    eg = np.frexp(np.abs(y).max() * slot_bound(g))[1]
    n = terms(g).reshape(ref.shape)
    # each term half a unit; the sum of an axis, the voxel's and the product y x length by one rounding each
    bar = n * 0.5 * 2.0 ** (eg - 62.0) + 3 * eps * mag * (1 + 1e-6)
    err = np.abs(np.asarray(got, np.float64) - ref)
    assert np.all(err <= bar), (err - bar).max()
    return bar, mag


@pytest.mark.parametrize("vol,det,s2c,c2d,angles", [
    ((10, 50, 9), (30, 120), 16.0, 8.0, (0.0, 40.0, 90.0, 200.0)),
    ((33, 40, 35), (50, 90), 40.0, 20.0, (0.0, 35.0, 100.0))], ids=str)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_three_driving_axes(vol, det, s2c, c2d, angles, dtype):
    import elsa_amd as E

    g = oracle.circle_geometry(3, vol, len(angles), 360, s2c, c2d, det=det, angles_deg=np.asarray(angles, np.float32))
    axis, nsteps = oracle.joseph_rays(g)[:2]
    assert len(np.unique(axis[nsteps > 0])) == 3
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(8).standard_normal(g.sino_shape).astype(dtype)
    got = op.applyAdjoint(y)
    f32 = dtype == np.float32
    check(got, g, y.astype(np.float64), oracle.MODE_EXACT_WEIGHTS if f32 else oracle.MODE_DIRECT,
          2.0 ** -24 if f32 else 2.0 ** -52)
    for tile in ((8, 17, 17), (4, 32, 32), (1, 1, 1), (3, 6, 5), (8, 22, 24)):
        op.tile(*tile)
        np.testing.assert_array_equal(op.applyAdjoint(y), got, err_msg=str(tile))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("det,poses", [(9, 7), (64, 512), (64, 513)])
def test_scale_of_small_2d_problems(det, poses, dtype):
    """With the largest value anywhere: a scale taken a few bits too coarse would show at the voxels that its ray
    does not meet."""
    import elsa_amd as E

    g = oracle.circle_geometry(2, (23, 17), poses, 360, 300.0, 100.0, det=(det,))
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    f32 = dtype == np.float32
    n = det * poses
    for k in (0, n // 2, n - 1):
        y = np.random.default_rng(k).random(g.sino_shape)
        y.reshape(-1)[k] = 2.0 ** 30
        y = y.astype(dtype)
        bar, mag = check(op.applyAdjoint(y), g, y.astype(np.float64),
                         oracle.MODE_EXACT_WEIGHTS if f32 else oracle.MODE_DIRECT, 2.0 ** -24 if f32 else 2.0 ** -52)
        # the bar tells: far below the sums of the ordinary values (some hundred over 512 poses)
        assert np.median(bar) < 1e-2

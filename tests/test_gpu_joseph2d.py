"""The 2D Joseph kernels at the edges of their tiles, pose steps and span parts, against the oracle:
volumes smaller than a tile, one row, remainders; tiles of every shape (also larger than the LDS
takes) with the same bits; more poses than a step takes; spans shorter than their parts; launches
of one, two and four parts, alone and in a batch; rays near 45 degrees."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors
from fp32_bounds import check_forward

pytestmark = pytest.mark.gpu

# vol, poses, detector, angles (None: a full circle)
CASES = [
    ((1, 5), 9, 12, None),
    ((16, 16), 7, 30, None),
    ((17, 33), 40, 60, None),
    ((31, 8), 23, 50, (43.0, 47.0)),
    ((70, 130), 64, 200, None),
    ((24, 24), 700, 40, None),  # two pose steps
]


def _geometry(case, dtype=np.float32):
    vol, poses, det, span = case
    angles = np.linspace(*(span or (0.0, 360.0)), poses).astype(np.float32)
    n = max(vol)
    return oracle.circle_geometry(2, vol, poses, 360, 20.0 * n, 4.0 * n, det=(det,), angles_deg=angles)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])) + "-%d" % c[1])
def test_back_projection(case, dtype):
    import elsa_amd as E

    g = _geometry(case)
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(3).standard_normal(g.sino_shape).astype(dtype)
    got = op.applyAdjoint(y)
    mode = oracle.MODE_EXACT_WEIGHTS if dtype == np.float32 else oracle.MODE_DIRECT
    ref = oracle.joseph(g, y.astype(np.float64), adjoint=True, mode=mode, acc64=True)
    mag = oracle.joseph(g, np.abs(y).astype(np.float64), adjoint=True, mode=mode, acc64=True)
    # FP32 rounds the product y * len of each term and the voxel; FP64 rounds the voxel and its terms
    # to a unit below 2^-44 of the largest slot sum possible
    eps = 2.0 ** -24 if dtype == np.float32 else 2.0 ** -52
    assert np.all(np.abs(got - ref) <= 2 * eps * mag * (1 + 1e-6) + 2.0 ** -44 * np.abs(y).max())
    for tile in ((8, 8), (5, 3), (32, 16), (1, 1), (200, 12)):
        op.tile(*tile)
        np.testing.assert_array_equal(op.applyAdjoint(y), got, err_msg=str(tile))
    for poses in (1, 3, 32):
        op.pose_batch(poses)
        np.testing.assert_array_equal(op.applyAdjoint(y), got, err_msg=f"{poses} poses")
    y.reshape(-1)[1] = np.inf
    assert np.isnan(op.applyAdjoint(y)).all()
    y.reshape(-1)[1] = 1.0  # and the exponent of the next call is its own
    y[:] = 0
    assert not op.applyAdjoint(y).any()


@pytest.mark.parametrize("case", CASES + [((9, 7), 8192, 70, None), ((5, 6), 9000, 20, None)],
                         ids=lambda c: "x".join(map(str, c[0])) + "-%d" % c[1])
def test_forward(case):
    import elsa_amd as E

    g = _geometry(case)
    ops = [E.JosephsMethodCUDA(*geom_to_descriptors(g)) for _ in range(2)]
    x = np.random.default_rng(4).standard_normal(g.vol_shape).astype(np.float32)
    got = ops[0].apply(x)
    check_forward(got, g, x)
    B = E.ProjectorBatch(ops)  # the parts one after another: the same sums
    fx = B.unpack(B.apply(B.pack([x, 2 * x])), adjoint_space=True)
    np.testing.assert_array_equal(fx[0].cpu().numpy(), got)
    np.testing.assert_array_equal(fx[1].cpu().numpy(), 2 * got)


def test_exponent_over_many_blocks():
    """The largest |y| decides the fixed-point unit wherever it lies: a back projection of y with one
    value a power of two above the rest moves with it."""
    import torch

    import elsa_amd as E

    g = _geometry(((40, 40), 300, 90, None))
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g))
    y = torch.zeros(g.sino_shape, device="cuda")
    base = None
    for at in (0, 4095, 4096, 13000, y.numel() - 1):
        y.zero_()
        y.view(-1)[at] = 1.0
        one = op.applyAdjoint(y).clone()
        y.view(-1)[at] = 2.0 ** 60
        np.testing.assert_array_equal((op.applyAdjoint(y) * 2.0 ** -60).cpu().numpy(), one.cpu().numpy())
        base = one if base is None else base
    y.zero_()
    y.view(-1)[0] = 1.0
    torch.testing.assert_close(op.applyAdjoint(y), base, rtol=0, atol=0)

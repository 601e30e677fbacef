"""The 3D Joseph back projection's launches against the oracle: rays of one driving axis, of two (both
axes' tiles in one launch) and of three, in every storage type, alone and in batches; volumes smaller
than a tile and with remainders; tiles of every shape with the same bits; voxels that one axis leaves
at zero."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors
from fp32_bounds import check_forward

pytestmark = pytest.mark.gpu

# vol, det, source and detector distance, angles: axes that drive rays
CASES = {
    "one": ((9, 33, 12), (20, 40), 400.0, 100.0, (0.0, 5.0, -7.0)),
    "two": ((17, 35, 40), (70, 50), 400.0, 100.0, tuple(range(0, 360, 24))),
    "two_small": ((1, 3, 2), (7, 6), 100.0, 50.0, (0.0, 30.0, 90.0, 45.0)),
    "three": ((10, 50, 9), (30, 120), 16.0, 8.0, (0.0, 40.0, 90.0, 200.0)),
}


def _geometry(name):
    vol, det, s2c, c2d, angles = CASES[name]
    return oracle.circle_geometry(3, vol, len(angles), 360, s2c, c2d, det=det,
                                  angles_deg=np.asarray(angles, np.float32))


@pytest.mark.parametrize("name,dtype", [(n, np.float32) for n in CASES] +
                         [(n, np.float64) for n in CASES if n != "three"], ids=str)
def test_back_projection(name, dtype):
    import elsa_amd as E

    g = _geometry(name)
    axis, nsteps = oracle.joseph_rays(g)[:2]
    assert len(np.unique(axis[nsteps > 0])) == {"one": 1, "three": 3}.get(name, 2)
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    y = np.random.default_rng(8).standard_normal(g.sino_shape).astype(dtype)
    got = op.applyAdjoint(y)
    mode = oracle.MODE_EXACT_WEIGHTS if dtype == np.float32 else oracle.MODE_DIRECT
    ref = oracle.joseph(g, y.astype(np.float64), adjoint=True, mode=mode, acc64=True)
    mag = oracle.joseph(g, np.abs(y).astype(np.float64), adjoint=True, mode=mode, acc64=True)
    # FP32 rounds the product y * len of each term, each axis' sum and the voxel; FP64 rounds its terms to
    # a unit below 2^-44 of the largest slot sum possible, and the sums
    eps = 2.0 ** -24 if dtype == np.float32 else 2.0 ** -52
    assert np.all(np.abs(got - ref) <= 3 * eps * mag * (1 + 1e-6) + 2.0 ** -44 * np.abs(y).max())
    for tile in ((8, 17, 17), (4, 32, 32), (1, 1, 1), (3, 6, 5), (8, 22, 24), (16, 8, 9)):
        op.tile(*tile)
        np.testing.assert_array_equal(op.applyAdjoint(y), got, err_msg=str(tile))
    y[:] = 0
    assert not op.applyAdjoint(y).any()


@pytest.mark.parametrize("vol", [(40, 6, 37), (284, 5, 9), (285, 5, 9), (9, 4, 330), (3, 300, 2)], ids=str)
def test_forward_of_short_and_long_rows(vol):
    """Four samples at once over view rows up to 2304 bytes (284 voxels), two over longer ones; spans that
    leave one to three samples over."""
    import elsa_amd as E

    n = max(vol)
    angles = np.array([0.0, 20.0, 45.0, 71.0, 90.0, 200.0], np.float32)
    g = oracle.circle_geometry(3, vol, len(angles), 360, 10.0 * n, 3.0 * n, det=(int(1.5 * n), 12),
                               angles_deg=angles)
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=np.float32)
    x = np.random.default_rng(12).standard_normal(g.vol_shape).astype(np.float32)
    check_forward(op.apply(x), g, x)


@pytest.mark.parametrize("names", [("two", "two_small", "one"), ("two", "three"), ("one", "one")])
def test_batch_equals_each_operator(names):
    import elsa_amd as E

    gs = [_geometry(n) for n in names]
    ops = [E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=np.float32) for g in gs]
    rng = np.random.default_rng(9)
    ys = [rng.standard_normal(g.sino_shape).astype(np.float32) for g in gs]
    batch = E.ProjectorBatch(ops)
    assert batch.fused
    out = batch.unpack(batch.applyAdjoint(batch.pack(ys, adjoint_space=True)))
    for got, op, y in zip(out, ops, ys):
        np.testing.assert_array_equal(got.cpu().numpy(), op.applyAdjoint(y))


def test_bf16_is_the_rounded_fp32_result():
    import torch

    import elsa_amd as E

    g = _geometry("two")
    y = torch.from_numpy(np.random.default_rng(10).standard_normal(g.sino_shape)).to(torch.bfloat16).cuda()
    low = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype="bfloat16")
    full = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=np.float32)
    assert torch.equal(low.applyAdjoint(y), full.applyAdjoint(y.float()).to(torch.bfloat16))

"""The fixed-point scale's max |y| finds the largest value wherever it lies and however the data are
aligned: a sinogram in the middle of a buffer gives the back projection of its aligned copy, bit for
bit, with the largest value at either end, next to the vector loads' edges and in the last block."""
import numpy as np
import pytest

import oracle
from backends import geom_to_descriptors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64", "bfloat16"])
@pytest.mark.parametrize("det,poses", [((1, 1), 1), ((7, 3), 1), ((128, 128), 1), ((131, 127), 1), ((300, 200), 18)])
def test_back_projection_of_unaligned_data(det, poses, dtype):
    import torch

    import elsa_amd as E

    g = oracle.circle_geometry(3, (6, 5, 7), poses, 360, 300.0, 100.0, det=det)
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    n = int(np.prod(g.sino_shape))
    t = getattr(torch, dtype)
    data = torch.randn(n, generator=torch.Generator().manual_seed(3)).to(t)
    for off in (0, 1, 2, 5):
        buf = torch.zeros(n + 16, dtype=t, device="cuda")
        for k in sorted({0, min(1, n - 1), n // 2, max(n - 5, 0), n - 1}):
            y = buf[off:off + n]
            y.copy_(data)
            y[k] = 2.0 ** 40
            got = op.applyAdjoint(y.view(g.sino_shape))
            assert torch.equal(got, op.applyAdjoint(y.clone().view(g.sino_shape))), (off, k)
            y[k] = float("nan")
            assert torch.isnan(op.applyAdjoint(y.view(g.sino_shape))).all(), (off, k)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("det,poses", [(9, 7), (64, 512), (64, 513)])
def test_small_2d_problems_find_it_in_their_tiles(det, poses, dtype):
    """Up to 32768 rays every tile of a 2D back projection finds the scale itself, past them a launch
    before it: the largest value counts wherever it lies (a smaller scale would overflow), unaligned data
    too, and an infinity makes every voxel NaN."""
    import torch

    import elsa_amd as E

    g = oracle.circle_geometry(2, (23, 17), poses, 360, 300.0, 100.0, det=(det,))
    op = E.JosephsMethodCUDA(*geom_to_descriptors(g), dtype=dtype)
    n = det * poses
    t = getattr(torch, dtype)
    buf = torch.zeros(n + 16, dtype=t, device="cuda")
    eps = 2.0 ** -24 if dtype == "float32" else 2.0 ** -52
    for off in (0, 3):
        y = buf[off:off + n].view(g.sino_shape)
        for k in (0, n // 2, n - 1):
            y.copy_(torch.rand(n, dtype=torch.float64, generator=torch.Generator().manual_seed(k)).view(g.sino_shape))
            y.view(-1)[k] = 2.0 ** 30
            got = op.applyAdjoint(y).double().cpu().numpy()
            ref = oracle.joseph(g, y.double().cpu().numpy(), adjoint=True, mode=oracle.MODE_EXACT_WEIGHTS, acc64=True)
            # rounding of the terms and the sum; n terms of half a unit, a unit below 2^-40 of the largest value
            assert np.all(np.abs(got - ref) <= 3 * eps * ref + n * 2.0 ** -41 * 2.0 ** 30 + 1e-6 * ref)
            y.view(-1)[k] = float("inf")
            assert torch.isnan(op.applyAdjoint(y)).all()

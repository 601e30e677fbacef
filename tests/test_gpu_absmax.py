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

"""3D Joseph forwards over tilted trajectories, whose views take four samples at once over rows of up to 800 or 1312
bytes and two over longer ones, against the oracle; spans that leave one to three samples over."""
import numpy as np
import pytest

from backends import GpuBackend, OracleBackend
from fp32_bounds import check_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vol", [(95, 6, 37), (96, 5, 9), (97, 5, 9), (9, 4, 130), (3, 110, 2), (160, 4, 7), (5, 3, 161)], ids=str)
@pytest.mark.parametrize("beta", [0.3, 1.5])
def test_forward_of_tilted_trajectories(vol, beta):
    import elsa_amd as E

    n = max(vol)
    poses = [dict(s2c=6.0 * n, c2d=2.0 * n, gamma=a, beta=beta * np.sin(2.0 * a + 0.5))
             for a in np.linspace(0.0, 5.5, 9)]
    det = (int(1.5 * n), 24)
    g = OracleBackend().setup(vol, det, poses)
    op = E.JosephsMethodCUDA(*GpuBackend().setup(vol, det, poses), dtype=np.float32)
    x = np.random.default_rng(12).standard_normal(g.vol_shape).astype(np.float32)
    check_forward(op.apply(x), g, x)

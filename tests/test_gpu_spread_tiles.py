"""2D matrix spreading with the longest tiles that it accepts.

A tile of 4 x 256 cells has records of 280 floats, and a staging round of 128
of them holds more floats than 15 bits count.  Against the cell-owner kernel
(1e-6, the bar between the spreading kernels) and the FP64 ES-NUFFT (1e-5).
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [(4, 256), (8, 128), (64, 16)], ids=str)
def test_long_tiles(tile):
    from hipnufft import _capi

    shape, T, M = (40, 300), 9, 8000
    om = (rand_traj(M, 2, 51) * np.float32(2 * np.pi)).astype(np.float32)
    om[: M // 2] *= 0.2  # full staging rounds in the central tiles
    k = rand_cplx((T, M), 52)
    got = []
    for method in (4, 1):  # matrix, cells
        plan = _capi.RawPlan(shape, n_trans=T, tile=tile, spread_method=method)
        plan.setpts(torch.from_numpy(om).cuda())
        z = torch.empty((T, *shape), dtype=torch.complex64, device="cuda")
        plan.sense_adj(torch.from_numpy(k).cuda(), None, None, z, T, 1, 1.0)
        got.append(z.cpu().numpy())
    assert rel_l2(got[0], got[1]) < 1e-6
    ref = nufft.Plan(om, shape)
    for t in (0, T - 1):
        assert rel_l2(got[0][t], ref.execute_adjoint(k[t])) < 1e-5

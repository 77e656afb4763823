"""Interpolation with 3D tiles far from the default 8 x 8 x 16.

Regions smaller than the point weights that are exchanged through the same
LDS.  Oracle: the FP64 ES-NUFFT of the same kernel width, 1e-5.
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,span,eps", [
    ((4, 4, 8), 1, 1e-3), ((4, 4, 8), 1, 1e-1), ((4, 4, 4), 2, 1e-3), ((2, 2, 2), 2, 1e-2),
], ids=str)
def test_tiles(tile, span, eps):
    from hipnufft import _capi

    shape, M, T = (20, 26, 22), 6000, 3
    traj = rand_traj(M, 3, 41)
    traj[: M // 2] *= 0.1  # full items in the central tiles
    om = (traj * np.float32(2 * np.pi)).astype(np.float32)
    plan = _capi.RawPlan(shape, n_trans=T, eps=eps, tile=tile, interp_span=span)
    plan.setpts(torch.from_numpy(om).cuda())
    x = rand_cplx((T, *shape), 42)
    y = torch.empty((T, M), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, T, 1, 1.0)
    ref = nufft.Plan(om, shape, eps=eps)
    for t in range(T):
        assert rel_l2(y[t].cpu().numpy(), ref.execute(x[t])) < 1e-5

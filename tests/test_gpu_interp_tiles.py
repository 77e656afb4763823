"""Interpolation with tiles far from the default ones.

Regions smaller than the point weights that are exchanged through the same
LDS, and rows of more 16-cell chunks than a chunk mask has bits (16), or than
a word has (32).  Oracle: the FP64 ES-NUFFT of the same kernel width, 1e-5.
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,tile,span,eps,max_sub", [
    ((20, 26, 22), (4, 4, 8), 1, 1e-3, 0), ((20, 26, 22), (4, 4, 8), 1, 1e-1, 0),
    ((20, 26, 22), (4, 4, 4), 2, 1e-3, 0), ((20, 26, 22), (2, 2, 2), 2, 1e-2, 0),
    ((10, 12, 160), (1, 1, 128), 2, 1e-3, 0), ((10, 12, 160), (1, 1, 128), 2, 1e-3, 200),
    ((10, 12, 300), (1, 1, 256), 2, 1e-2, 0), ((10, 12, 300), (1, 1, 256), 2, 1e-2, 200),
    ((10, 300), (1, 512), 1, 1e-3, 0),
], ids=str)
def test_tiles(shape, tile, span, eps, max_sub):
    from hipnufft import _capi

    M, T, D = 6000, 3, len(shape)
    traj = rand_traj(M, D, 41)
    traj[: M // 2] *= 0.1  # full items in the central tiles
    om = (traj * np.float32(2 * np.pi)).astype(np.float32)
    plan = _capi.RawPlan(shape, n_trans=T, eps=eps, tile=tile, interp_span=span,
                          max_subproblem=max_sub)
    plan.setpts(torch.from_numpy(om).cuda())
    x = rand_cplx((T, *shape), 42)
    y = torch.empty((T, M), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, T, 1, 1.0)
    ref = nufft.Plan(om, shape, eps=eps)
    for t in range(T):
        assert rel_l2(y[t].cpu().numpy(), ref.execute(x[t])) < 1e-5

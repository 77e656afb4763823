"""Transforms on grids of the lengths with compile-time FFT plans, and others.

Every compile-time length on both kinds of axis, one image (workgroups of few
lines) and many, radix 10 on its own and after 8s, and lengths that take the
runtime plans.  Adjointness to 1e-5 and parity with the FP64 oracle NUFFT to
1e-5 (eps = 1e-6).
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 40])
@pytest.mark.parametrize("shape", [
    (64, 96), (96, 64), (128, 160), (160, 128), (192, 256), (256, 192), (320, 384), (384, 320),
    (40, 125), (125, 20), (10, 45), (75, 90),
], ids=str)
def test_lengths(shape, T):
    from hipnufft import _capi

    M = 500
    om = (rand_traj(M, 2, 21) * np.float32(2 * np.pi)).astype(np.float32)
    plan = _capi.RawPlan(shape, n_trans=T)
    plan.setpts(torch.from_numpy(om).cuda())
    x, k = rand_cplx((T, *shape), 22), rand_cplx((T, M), 23)
    y = torch.empty((T, M), dtype=torch.complex64, device="cuda")
    z = torch.empty((T, *shape), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, T, 1, 1.0)
    plan.sense_adj(torch.from_numpy(k).cuda(), None, None, z, T, 1, 1.0)
    y, z = y.cpu().numpy(), z.cpu().numpy()
    ref = nufft.Plan(om, shape)
    for t in {0, T - 1}:
        assert rel_l2(y[t], ref.execute(x[t])) < 1e-5
        assert rel_l2(z[t], ref.execute_adjoint(k[t])) < 1e-5
    assert abs(np.vdot(k, y) - np.vdot(z, x)) < 1e-5 * np.linalg.norm(k) * np.linalg.norm(y)

"""Axes whose runtime FFT plan has a radix-10 pass, and the kernels' own
instances for them: 50, 80, 250 and 400 points on every kind of axis, one
image (workgroups of few lines) and many, the Toeplitz middle pass and the
stacked z axis.  Oracles: the FP64 ES-NUFFT and the FP64 stacked operator
(1e-5, eps = 1e-6), and adj_op(op) for the Toeplitz form (2e-5, the bar of
the other lengths).
"""

import numpy as np
import pytest
import torch

from helpers import gauss_smaps, radial2d, rand_cplx, rand_traj, rel_l2
from oracle import nufft
from oracle import stacked as ost

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,T", [
    ((200, 40), 1), ((200, 40), 30), ((25, 200), 1), ((25, 200), 30), ((125, 25), 30),
    ((200, 24, 40), 1), ((25, 40, 200), 2),
], ids=str)
def test_transforms(shape, T):
    from hipnufft import _capi

    M, D = 600, len(shape)
    om = (rand_traj(M, D, 61) * np.float32(2 * np.pi)).astype(np.float32)
    plan = _capi.RawPlan(shape, n_trans=T)
    plan.setpts(torch.from_numpy(om).cuda())
    x, k = rand_cplx((T, *shape), 62), rand_cplx((T, M), 63)
    y = torch.empty((T, M), dtype=torch.complex64, device="cuda")
    z = torch.empty((T, *shape), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, T, 1, 1.0)
    plan.sense_adj(torch.from_numpy(k).cuda(), None, None, z, T, 1, 1.0)
    ref = nufft.Plan(om, shape)
    for t in {0, T - 1}:
        assert rel_l2(y[t].cpu().numpy(), ref.execute(x[t])) < 1e-5
        assert rel_l2(z[t].cpu().numpy(), ref.execute_adjoint(k[t])) < 1e-5


@pytest.mark.parametrize("shape", [(200, 40), (40, 25, 20)], ids=str)
def test_toeplitz(shape):
    import hipnufft

    op = hipnufft.get_operator("hipnufft")(rand_traj(900, len(shape), 64), shape, n_coils=3,
                                           smaps=gauss_smaps(3, shape, 65))
    op.compute_toeplitz_kernel()
    x = torch.from_numpy(rand_cplx((1, 1, *shape), 66)).cuda()
    assert rel_l2(op.gram_op(x).cpu().numpy(), op.adj_op(op.op(x)).cpu().numpy()) < 2e-5


@pytest.mark.parametrize("Z", [10, 80, 250, 400])
def test_stacked(Z):
    import hipnufft

    s2, shape, C = radial2d(8, 20), (12, 14, Z), 2
    smaps = gauss_smaps(C, shape, 67)
    zi = np.arange(Z)
    op = hipnufft.get_operator("stacked-hipnufft")(s2, shape, smaps=smaps, n_coils=C, z_index=zi)
    x, k = rand_cplx((1, *shape), 68), rand_cplx((1, C, op.n_samples), 69)
    yref = ost.op(s2, zi, x, shape, smaps)
    zref = ost.adj(s2, zi, k, shape, smaps)
    assert rel_l2(np.asarray(op.op(x)).reshape(yref.shape), yref) < 1e-5
    assert rel_l2(np.asarray(op.adj_op(k)).reshape(zref.shape), zref) < 1e-5

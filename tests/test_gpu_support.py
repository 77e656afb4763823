"""Transforms whose points leave part of the fine grid untouched.

Tiles that no footprint touches are neither written nor read.  Each case
first fills the plan's whole workspace with NaN (points everywhere, a NaN
image), then moves to points that cover only part of k-space, with lines
and whole tiles outside: any stale cell that is still read shows.  Tiles of
other sizes, several point sets with different supports, no points at all,
and axes that do not divide into a wave's positions.  Oracle: the FP64
ES-NUFFT, 1e-5 (eps = 1e-6).
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


def _points(kind, M, D, seed):
    x = 2 * np.pi * rand_traj(M, D, seed).astype(np.float64)
    if kind == "ball":
        x *= (np.pi / np.maximum(np.linalg.norm(x, axis=1), np.pi))[:, None]
    elif kind == "corner":  # wraps around the origin of the grid
        x *= 0.12
    elif kind == "line":
        x[:, 1:] = 0.4
    return np.clip(x, -np.pi, np.nextafter(np.pi, 0)).astype(np.float32)


def _poison(plan, shape, T):
    plan.setpts(torch.from_numpy(_points("all", 20000, len(shape), 1)).cuda())
    x = torch.full((T, *shape), float("nan"), dtype=torch.complex64, device="cuda")
    y = torch.empty((T, 20000), dtype=torch.complex64, device="cuda")
    plan.sense_op(x, None, y, T, 1, 1.0)
    plan.sense_adj(y, None, None, x, T, 1, 1.0)


@pytest.mark.parametrize("kind", ["ball", "corner", "line", "all"])
@pytest.mark.parametrize("shape,opts", [
    ((48, 40, 44), {}), ((29, 33, 31), {}), ((96, 64), {}), ((75, 90), {}),
    ((96, 64), {"tile": (16, 16)}), ((40, 36, 32), {"tile": (4, 8, 16)}),
    ((40, 36, 32), {"tile": (16, 8, 8), "spread_method": 1}), ((300, 40), {"tile": (2, 32)}),
], ids=str)
def test_partial_support(shape, opts, kind):
    from hipnufft import _capi

    T, M = 3, 700
    plan = _capi.RawPlan(shape, n_trans=T, **opts)
    _poison(plan, shape, T)
    om = _points(kind, M, len(shape), 2)
    plan.setpts(torch.from_numpy(om).cuda())
    x, k = rand_cplx((T, *shape), 3), rand_cplx((T, M), 4)
    y = torch.empty((T, M), dtype=torch.complex64, device="cuda")
    z = torch.empty((T, *shape), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, T, 1, 1.0)
    plan.sense_adj(torch.from_numpy(k).cuda(), None, None, z, T, 1, 1.0)
    ref = nufft.Plan(om, shape)
    for t in range(T):
        assert rel_l2(y[t].cpu().numpy(), ref.execute(x[t])) < 1e-5
        assert rel_l2(z[t].cpu().numpy(), ref.execute_adjoint(k[t])) < 1e-5


def test_sets_with_different_supports():
    from hipnufft import _capi

    shape, kinds, M = (64, 48), ["corner", "ball", "line"], [300, 900, 50]
    plan = _capi.RawPlan(shape, n_trans=6)
    _poison(plan, shape, 6)
    oms = [_points(k, m, 2, 5 + m) for k, m in zip(kinds, M)]
    plan.setpts_sets([torch.from_numpy(o).cuda() for o in oms])
    x = rand_cplx((3, 2, *shape), 6)
    k = [rand_cplx((2, m), 7 + m) for m in M]
    y = torch.empty(2 * sum(M), dtype=torch.complex64, device="cuda")
    z = torch.empty((3, 2, *shape), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, 3, 2, 1.0)
    kf = torch.from_numpy(np.concatenate([v.ravel() for v in k])).cuda()
    plan.sense_adj(kf, None, None, z, 3, 2, 1.0)
    y = np.split(y.cpu().numpy(), np.cumsum([2 * m for m in M])[:-1])
    for s in range(3):
        ref = nufft.Plan(oms[s], shape)
        for c in range(2):
            assert rel_l2(y[s].reshape(2, -1)[c], ref.execute(x[s, c])) < 1e-5
            assert rel_l2(z[s, c].cpu().numpy(), ref.execute_adjoint(k[s][c])) < 1e-5


@pytest.mark.parametrize("shape", [(48, 40, 44), (96, 64)], ids=str)
def test_no_points(shape):
    from hipnufft import _capi

    plan = _capi.RawPlan(shape, n_trans=2)
    _poison(plan, shape, 2)
    plan.setpts(torch.empty((0, len(shape)), device="cuda"))
    z = torch.full((2, *shape), float("nan"), dtype=torch.complex64, device="cuda")
    k = torch.empty((2, 1), dtype=torch.complex64, device="cuda")
    plan.sense_adj(k, None, None, z, 2, 1, 1.0)
    assert not z.cpu().numpy().any()

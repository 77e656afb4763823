"""Interpolation by aligned pairs of cells, at its edges.

A footprint row is read as the aligned pairs that cover it, one cell more
than the footprint: what stands there must not matter, not even an infinity
(spread / interp-only plans take the caller's grid as it is).  Grids whose
last axis is odd or whose memory is not 16-byte aligned are read cell by
cell; items of more than 128 points and tiny wrapped grids take the other
kernels.  Oracle: the FP64 ES-NUFFT (1e-5, the bar of the other transforms),
and the grid without the infinities (1e-6: the same sums, rounded alike).
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "8-byte-aligned"])
@pytest.mark.parametrize("start", [5, 8, 0])
@pytest.mark.parametrize("shape", [(48, 40, 44), (48, 40, 45), (48, 44), (48, 45)], ids=str)
def test_cells_outside_the_footprint(shape, start, shift):
    from hipnufft import _capi

    D, nf = len(shape), shape[-1]
    rng = np.random.default_rng(3)
    M, W = 150, 7
    x = rng.uniform(-np.pi, np.pi, (M, D)).astype(np.float32)
    x[:, -1] = 2 * np.pi * (start + W / 2 - 0.3) / nf  # every footprint starts at cell `start`
    plan = _capi.RawPlan(shape, n_trans=1, eps=1e-6, spreadinterponly=True)
    plan.setpts(torch.from_numpy(x).cuda())
    assert plan.info()["w"] == W
    n = int(np.prod(shape))
    clean = torch.from_numpy(rand_cplx(shape, 7)).cuda().reshape(-1)
    out = []
    for poison in (False, True):
        mem = torch.empty(n + 2, dtype=torch.complex64, device="cuda")
        grid = mem[shift:shift + n]
        grid.copy_(clean)
        if poison:
            g = grid.view(shape)
            for c in (start - 1, start + W):
                g[..., c % nf] = complex(float("inf"), float("nan"))
        y = torch.empty(M, dtype=torch.complex64, device="cuda")
        plan.sense_op(grid, None, y, 1, 1, 1.0)
        out.append(y.cpu().numpy())
    assert np.isfinite(out[1]).all()
    assert rel_l2(out[1], out[0]) < 1e-6


@pytest.mark.parametrize("eps", [1e-1, 1e-2, 1e-3, 1e-4, 1e-5, 1e-6, 1e-7])
@pytest.mark.parametrize("shape,M,max_sub", [
    ((20, 26, 22), 3000, 0), ((20, 26, 22), 900, 200), ((7, 5, 9), 400, 0), ((40, 34), 5000, 0),
], ids=str)
def test_interp_widths(shape, M, max_sub, eps):
    from hipnufft import _capi

    traj = rand_traj(M, len(shape), 11)
    traj[: M // 2] *= 0.1  # several items in the central tiles
    om = (traj * np.float32(2 * np.pi)).astype(np.float32)
    plan = _capi.RawPlan(shape, n_trans=3, eps=eps, max_subproblem=max_sub)
    plan.setpts(torch.from_numpy(om).cuda())
    x = rand_cplx((3, *shape), 12)
    y = torch.empty((3, M), dtype=torch.complex64, device="cuda")
    plan.sense_op(torch.from_numpy(x).cuda(), None, y, 3, 1, 1.0)
    ref = nufft.Plan(om, shape, eps=eps)
    for t in range(3):
        assert rel_l2(y[t].cpu().numpy(), ref.execute(x[t])) < 1e-5

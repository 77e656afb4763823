"""The matrix spreading kernel's stores into grids of any shape and alignment.

Spread / interp-only plans spread into the caller's grid: rows of odd length
and grids that are not 16-byte aligned are stored cell by cell, the others in
pairs.  Against the cell-owner kernel (1e-6, the bar between the spreading
kernels), whole and split tiles, with the cells around the grids untouched.
"""

import numpy as np
import pytest
import torch

from helpers import rand_cplx, rand_traj, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [0, 32], ids=["whole", "split"])
@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "8-byte-aligned"])
@pytest.mark.parametrize("shape", [(45, 41, 37), (24, 20, 38), (50, 45), (70, 66)], ids=str)
def test_stores(shape, shift, split):
    from hipnufft import _capi

    T, M, n = 11, 900, int(np.prod(shape))
    x = 2 * np.pi * rand_traj(M, len(shape), 1).astype(np.float32)
    x[: M // 2] *= 0.1
    k = torch.from_numpy(rand_cplx((T, M), 2)).cuda()
    got = []
    for method in (4, 1):  # matrix, cells
        plan = _capi.RawPlan(shape, n_trans=T, spreadinterponly=True, spread_max=split,
                             spread_method=method)
        plan.setpts(torch.from_numpy(x).cuda())
        lo = 2 + shift
        mem = torch.full((T * n + 6,), 7.0, dtype=torch.complex64, device="cuda")
        plan.sense_adj(k, None, None, mem[lo:lo + T * n], T, 1, 1.0)
        out = mem.cpu().numpy()
        assert (out[:lo] == 7.0).all() and (out[lo + T * n:] == 7.0).all()
        got.append(out[lo:lo + T * n])
    assert rel_l2(got[0], got[1]) < 1e-6

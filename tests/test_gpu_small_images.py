"""Images with few rows: the coil sum of the adjoint's last-axis pass.

Few rows put several coils of a row side by side in a workgroup; the cases
hold row counts and coil counts that do not divide its lines, one coil, and
images whose coils span two chunks.  Parity with the FP64 oracle NUFFT, the
1e-5 bar of the other adjoint tests (eps = 1e-6).
"""

import numpy as np
import pytest
import torch

from helpers import gauss_smaps, rand_cplx, rand_traj, rel_l2
from oracle import nufft

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,coils,n_trans", [
    ((37, 50), 1, None), ((37, 50), 5, None), ((64, 48), 17, None), ((64, 64), 6, 3),
    ((21, 256), 3, None), ((5, 7, 30), 5, None), ((128,), 3, None),
], ids=lambda v: str(v))
def test_adjoint_coil_sum(shape, coils, n_trans):
    import hipnufft

    traj = rand_traj(1500, len(shape), 3)
    smaps = gauss_smaps(coils, shape, 4)
    op = hipnufft.get_operator("hipnufft")(traj, shape, n_coils=coils, smaps=smaps,
                                           n_trans=n_trans)
    y = rand_cplx((1, coils, len(traj)), 5)
    got = op.adj_op(torch.from_numpy(y).cuda()).cpu().numpy().reshape(shape)
    ref = nufft.Plan((traj * np.float32(2 * np.pi)).astype(np.float32), shape)
    want = sum(np.conj(smaps[c]) * ref.execute_adjoint(y[0, c]) for c in range(coils))
    assert rel_l2(got, want * op.inv_norm_factor) < 1e-5

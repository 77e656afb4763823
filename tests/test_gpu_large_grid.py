"""Transforms whose fine grid is just under 4 GiB or above it, where the cell
offsets of the strided FFT passes come near or pass 32 bits.  Oracle: the
exact sums in 64 bits at all samples and at random voxels, 1e-5 (eps = 1e-6,
the bar of the 192^3 headline).
"""

import pytest
import torch

import ndft_gpu

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(torch.linalg.vector_norm(a.to(b.dtype) - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("shape", [(400, 400, 400), (320, 512, 400), (420, 420, 420)], ids=str)
def test_large_grid(shape):
    from hipnufft import _capi

    M = 1000
    g = torch.Generator(device="cuda").manual_seed(31)
    om = (torch.rand((M, 3), generator=g, device="cuda") * 2 - 1) * 3.14159
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.complex64)
    k = torch.randn(M, generator=g, device="cuda", dtype=torch.complex64)
    plan = _capi.RawPlan(shape)
    plan.setpts(om)
    y, z = torch.empty_like(k), torch.empty_like(x)
    plan.sense_op(x, None, y, 1, 1, 1.0)
    plan.sense_adj(k, None, None, z, 1, 1, 1.0)
    torch.cuda.synchronize()
    assert _rel(y, ndft_gpu.type2(om, x, shape, chunk=256)[0]) < 1e-5
    vox = torch.randint(x.numel(), (2000,), generator=g, device="cuda")
    assert _rel(z.reshape(-1)[vox], ndft_gpu.type1_at(om, k, shape, vox)[0]) < 1e-5

"""The matmul kernel whose workgroup shares a 64 x 64 tile (matmul.hip: fp32 at block sizes 64 and above, 16-bit elements at
128 and above) where its loops can go wrong: no pair at all, one pair, lists longer than the 64 entries of a window, one
and several tiles per block, both operands read as they lie and transposed."""

import pytest
import torch

import blksprs_amd as bs
from oracle import blksprs_oracle as orc
from tests.helpers import assert_close, rand_blocks, rand_layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,sbs", [(torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 128),
                                       (torch.float16, 128), (torch.bfloat16, 256)])
@pytest.mark.parametrize("R,K,C,density", [(1, 1, 1, 1.0), (3, 2, 5, 0.3), (2, 70, 1, 1.0), (1, 1, 66, 1.0)])
def test_quad_kernel(device, dtype, sbs, R, K, C, density):
    B = 2
    lx, ly = rand_layout((B, R, K), density, 1, ensure_rows=True), rand_layout((B, K, C), density, 2, ensure_rows=True)
    lo = torch.ones((B, R, C), dtype=torch.bool)  # blocks without a pair become zeros
    x = rand_blocks(int(lx.sum()), sbs, dtype, 3, (K * sbs) ** -0.5)
    y = rand_blocks(int(ly.sum()), sbs, dtype, 4)
    go = rand_blocks(int(lo.sum()), sbs, dtype, 5, (max(R, C) * sbs) ** -0.5)
    xd, yd = (t.to(device).requires_grad_(True) for t in (x, y))
    out = bs.ops.matmul(xd, lx.to(device), yd, ly.to(device), lo.to(device), sbs)
    x64, y64 = (t.double().requires_grad_(True) for t in (x, y))
    ref = orc.matmul(x64, lx.numpy(), y64, ly.numpy(), lo.numpy(), sbs, acc_dtype=torch.float64)
    tol = 2e-5 if dtype == torch.float32 else 2e-2
    assert_close(out, ref, tol, "out")
    out.backward(go.to(device))
    ref.backward(go.double())
    assert_close(xd.grad, x64.grad, tol, "dX")
    assert_close(yd.grad, y64.grad, tol, "dY")

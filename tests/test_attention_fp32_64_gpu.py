"""fp32 attention in blocks of 64 on the kernels that take them as halves of 32 (attn_small_fwd.hip, attn_small_bwd.hip): one
and two head slices, lists that end within and at a window of 64 halves, masks, bias and causal lengths whose blocks are
read by quarters; slices that are missing and tensors that do not start on 16 bytes stay with the kernels before."""

import pytest
import torch

from tests.test_attention_gpu import _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh", [1, 2])
@pytest.mark.parametrize("use_mask,use_bias,use_causal", [(False, False, False), (True, False, False), (False, True, False),
                                                          (False, False, True), (True, True, True)])
def test_quarters(device, nh, use_mask, use_bias, use_causal):
    for B, n in ((1, 1), (3, 4), (9, 3)):
        _run_case(device, torch.float32, 64, B=B, nq=n, nk=n, nh=nh, nhv=nh, density=0.6, seed=10 * n + B, use_mask=use_mask,
                  use_bias=use_bias, use_causal=use_causal)


@pytest.mark.parametrize("nh", [1, 2])
@pytest.mark.parametrize("nk", [1, 2, 31, 32, 33, 70])
def test_list_lengths(device, nh, nk):
    _run_case(device, torch.float32, 64, B=1, nq=2, nk=nk, nh=nh, nhv=nh, density=1.0, seed=nk)
    _run_case(device, torch.float32, 64, B=2, nq=3, nk=nk, nh=nh, nhv=nh, density=0.3, seed=nk + 1, use_mask=True)


@pytest.mark.parametrize("nh,nhv", [(1, 2), (2, 2)])
def test_missing_slices(device, nh, nhv):
    _run_case(device, torch.float32, 64, B=2, nq=4, nk=5, nh=nh, nhv=nhv, density=0.5, seed=nh, use_mask=True,
              sparse_heads=True)
    _run_case(device, torch.float32, 64, B=2, nq=4, nk=5, nh=nh, nhv=nhv, density=0.5, seed=nh + 5, custom_o=True)

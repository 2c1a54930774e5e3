"""What the kernels for blocks of 16 and 32 leave to the fp32 matrix-core kernels that load through registers
(attn_f32mma.hip, attn_f32mma_bwd.hip): scales that are not positive, and head dimensions of q and k above 128 with at
most four value slices.  Every number of value slices those are built for and three of them, which run on the kernel for four."""

import pytest
import torch

from tests.test_attention_gpu import _run_case

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


# a bound: at |scale| <= 0.2 and up to 64 head dimensions scores are below 8, as with the scales of test_attention_gpu.py
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sbs,nh,nhv", [(16, 1, 1), (16, 4, 2), (16, 2, 3), (16, 3, 4), (32, 1, 1), (32, 2, 2), (32, 2, 3), (32, 1, 4)])
@pytest.mark.parametrize("scale", [-0.2, 0.0])
def test_scales_that_are_not_positive(device, dtype, sbs, nh, nhv, scale):
    """Full and sparse head layouts, lists longer than the four groups of waves take at once, bias, mask, causal lengths."""
    seed = 10 * nh + nhv
    _run_case(device, dtype, sbs, B=2, nq=4, nk=9, nh=nh, nhv=nhv, density=0.7, seed=seed, scale=scale)
    _run_case(device, dtype, sbs, B=2, nq=5, nk=5, nh=nh, nhv=nhv, density=0.6, seed=seed + 1, scale=scale, use_mask=True,
              use_bias=True, use_causal=True, sparse_heads=True, custom_o=True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sbs,nh,nhv", [(16, 9, 1), (16, 10, 4), (32, 5, 2), (32, 6, 3)])
def test_long_head_dimensions_of_queries_and_keys(device, dtype, sbs, nh, nhv):
    _run_case(device, dtype, sbs, B=2, nq=4, nk=9, nh=nh, nhv=nhv, density=0.6, seed=nh)
    _run_case(device, dtype, sbs, B=2, nq=5, nk=5, nh=nh, nhv=nhv, density=0.6, seed=nh + 1, use_mask=True, use_bias=True,
              use_causal=True, sparse_heads=True, custom_o=True)

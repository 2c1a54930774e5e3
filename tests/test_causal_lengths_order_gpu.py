"""Lengths beyond the range are refused ahead of everything that a call looks at after them."""

import pytest
import torch

import blksprs_amd as bs
from tests.helpers import rand_blocks

pytestmark = pytest.mark.gpu

SBS, N = 16, 4


def _call(device, lengths, **other):
    full, layout = (torch.ones((2, N, n), dtype=torch.bool, device=device) for n in (1, N))
    q, k, v = (rand_blocks(2 * N, SBS, torch.float32, seed).to(device) for seed in range(3))
    return bs.ops.flash_attention(q, full, k, full, v, full, layout, SBS, causal_lengths=lengths, **other)


@pytest.mark.parametrize("checking", [True, False])
@pytest.mark.parametrize("what,error", [("scale", TypeError), ("mask", ValueError), ("bias", ValueError), ("layout", ValueError)])
def test_lengths_come_first(device, what, error, checking):
    blocks = torch.zeros((1, SBS, SBS), device=device)
    other = {"scale": dict(scale="1"), "mask": dict(attention_mask=blocks), "bias": dict(attention_bias=blocks),
             "layout": dict(sparsity_layout_o=torch.ones((2, N + 1, 1), dtype=torch.bool, device=device))}[what]
    if not checking:
        bs.utils.disable_validation()
    try:
        for bad in (-1, N * SBS + 1):
            with pytest.raises(ValueError, match="causal_lengths values must be between zero and 64"):
                _call(device, torch.tensor([3, bad], device=device), **other)
        if checking or what != "layout":
            with pytest.raises(error) as seen:
                _call(device, torch.tensor([3, 7], device=device), **other)
            assert "causal_lengths" not in str(seen.value)
    finally:
        bs.utils.enable_validation()
    assert _call(device, torch.tensor([3, 7], device=device)).shape == (2 * N, SBS, SBS)

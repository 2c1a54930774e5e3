"""When the tables of shares (attn_shares.hip) are built: once per side of a layout, and for a call without a cache only where that
call gains by it."""

import pytest
import torch

import blksprs_amd as bs
from blksprs_amd import _capi
from tests.helpers import rand_blocks

pytestmark = pytest.mark.gpu


def _call(device, dtype, sbs, layout, full, cache, train):
    ops = [rand_blocks(full.numel(), sbs, dtype, seed).to(device).requires_grad_(train) for seed in range(3)]
    out = bs.ops.flash_attention(ops[0], full, ops[1], full, ops[2], full, layout, sbs, layout_cache=cache)
    return [out.detach(), *(torch.autograd.grad(out.sum(), ops) if train else ())]


def _long_rows(device, n):
    layout = torch.eye(n, dtype=torch.bool, device=device)[None].repeat(2, 1, 1)
    layout[:, 0] = True
    layout[:, :, 3] = True
    return layout, torch.ones((2, n, 1), dtype=torch.bool, device=device)


@pytest.fixture
def built(monkeypatch):
    """The sides (0: query rows, 1: key rows) of the tables that are built."""
    sides, call = [], _capi.call
    monkeypatch.setattr(_capi, "call", lambda name, *args: (sides.append(args[1]) if name == "bsa_attn_shares_build" else None,
                                                            call(name, *args))[1])
    return sides


@pytest.mark.parametrize("first", [False, True])
def test_one_cache_for_inference_and_training(device, built, first):
    layouts, cache = _long_rows(device, 260), {}  # a cache is for these tensors
    for train in (first, not first, first):
        _call(device, torch.bfloat16, 16, *layouts, cache, train)
    assert sorted(built) == [0, 1]
    shares = cache["tables"].shares
    assert shares[(16, torch.bfloat16, True)][0] is shares[(16, torch.bfloat16, False)][0] is not None


def test_calls_without_a_cache(device, built):
    layouts = _long_rows(device, 260)
    without = _call(device, torch.bfloat16, 16, *layouts, None, True)
    assert built == []
    for got, want in zip(without, _call(device, torch.bfloat16, 16, *layouts, {}, True)):
        assert float((got.double() - want.double()).norm() / want.double().norm()) < 1e-2
    assert built == [0, 1]
    _call(device, torch.float32, 32, *_long_rows(device, 130), None, True)
    assert built == [0, 1, 0, 1]

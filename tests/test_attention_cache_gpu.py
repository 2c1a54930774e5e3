"""A layout cache of attention that has been used: copied, and on the short way that a call with validation off takes through it."""

import copy
import gc

import pytest
import torch

import blksprs_amd as bs
from oracle import blksprs_oracle as orc
from tests.helpers import rand_blocks, rand_layout

pytestmark = pytest.mark.gpu


class _Layer(torch.nn.Module):
    """What a program keeps: layouts and the cache for them."""

    def __init__(self, device, sbs, uneven, seed=0, B=2, n=6, slices=2):
        super().__init__()
        if uneven:  # two rows and a column of all blocks: their walks are shared
            layout = torch.eye(n, dtype=torch.bool)[None].repeat(B, 1, 1)
            layout[:, 0] = layout[:, :, 3] = True
        else:
            layout = rand_layout((B, n, n), 0.5, seed, ensure_rows=True)
        self.sbs, self.cache = sbs, {}
        self.register_buffer("layout", layout.to(device))
        self.register_buffer("full", torch.ones((B, n, slices), dtype=torch.bool, device=device))

    def inputs(self, dtype, seed):
        return [rand_blocks(self.full.numel(), self.sbs, dtype, seed + i) for i in range(4)]

    def forward(self, q, k, v, **extra):
        return bs.ops.flash_attention(q, self.full, k, self.full, v, self.full, self.layout, self.sbs,
                                      layout_cache=self.cache, **extra)


def _results(layer, blocks, **extra):
    device = layer.layout.device
    q, k, v = (b.to(device).requires_grad_(True) for b in blocks[:3])
    out = layer(q, k, v, **extra)
    return [out.detach(), *torch.autograd.grad(out, (q, k, v), blocks[3].to(device))]


def _assert_as_oracle(layer, blocks, got, tol=4e-6):
    """fp32 operands: 32-bit sums leave 5e-7 to 9e-7 of the norm."""
    q, k, v = (b.double().requires_grad_(True) for b in blocks[:3])
    full, layout = layer.full.cpu().numpy(), layer.layout.cpu().numpy()
    out = orc.flash_attention(q, full, k, full, v, full, layout, layer.sbs, acc_dtype=torch.float64)
    want = [out.detach(), *torch.autograd.grad(out, (q, k, v), blocks[3].double())]
    for g, w in zip(got, want):
        assert float((g.double().cpu() - w).norm()) <= tol * float(w.norm())


@pytest.fixture(params=[True, False], ids=["checked", "unchecked"])
def validation(request):
    if not request.param:
        bs.utils.disable_validation()
    yield request.param
    bs.utils.enable_validation()


@pytest.mark.parametrize("sbs,n,uneven", [(64, 6, False), (32, 6, False), (32, 130, True)])
def test_a_layer_with_a_used_cache_is_copied(device, validation, sbs, n, uneven):
    layer = _Layer(device, sbs, uneven, n=n, slices=1 if uneven else 2)
    blocks = layer.inputs(torch.float32, 1)
    first = _results(layer, blocks)
    copied = copy.deepcopy(layer)
    del layer
    gc.collect()
    overwritten = [torch.full((1 << 16,), -1, dtype=torch.int32, device=device) for _ in range(64)]
    for _ in range(2):
        for got, want in zip(_results(copied, blocks), first):
            assert torch.equal(got, want)
    _assert_as_oracle(copied, blocks, first)
    del overwritten

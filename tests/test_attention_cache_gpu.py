"""A layout cache of attention that has been used: copied, and on the short way that a call with validation off takes through it."""

import copy
import gc
import threading

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


def _fresh(layer, blocks, **extra):
    kept, layer.cache = layer.cache, {}
    results = _results(layer, blocks, **extra)
    layer.cache = kept
    return results


def _assert_same(got, want):
    assert all(torch.equal(g, w) for g, w in zip(got, want))


def test_one_cache_for_layouts_of_several_sizes(device, validation):
    layers = [_Layer(device, sbs, False, seed=n, n=n) for sbs, n in ((32, 6), (32, 5), (64, 6), (64, 4))]
    for layer in layers:
        layer.cache = layers[0].cache
    for layer in (*layers, *layers[::-1], layers[0]):
        blocks = layer.inputs(torch.float16, 3)
        want = _fresh(layer, blocks)
        for _ in range(2):
            _assert_same(_results(layer, blocks), want)


@pytest.mark.parametrize("sbs", [32, 64])
@pytest.mark.parametrize("meddle", [
    lambda cache: cache.pop("key_indices_i32"),
    lambda cache: cache.pop("tables"),
    lambda cache: cache.pop("packed_indices_v"),
    lambda cache: cache.update(packed_indices_q=torch.zeros_like(cache["packed_indices_q"])),
    lambda cache: cache.update(tables=object()),
    lambda cache: cache["query_indices_i32"].zero_(),
    lambda cache: cache.update(of_the_caller=1),
], ids=["without_indices", "without_tables", "without_packed", "other_packed", "other_tables", "written_indices", "added"])
def test_a_cache_that_was_meddled_with_is_made_again(device, validation, sbs, meddle):
    layer = _Layer(device, sbs, False)
    blocks = layer.inputs(torch.float16, 5)
    want = _results(layer, blocks)
    meddle(layer.cache)
    for _ in range(2):
        _assert_same(_results(layer, blocks), want)


@pytest.mark.parametrize("sbs", [32, 64])
def test_masks_in_turn_on_one_cache(device, validation, sbs):
    """Blocks of 64: the lists without the pairs that a mask rules out take the place of the tables' own for that mask only."""
    layer = _Layer(device, sbs, False)
    blocks = layer.inputs(torch.bfloat16, 7)
    count = int(layer.layout.sum())
    masks = [(torch.rand((count, 1, 1), device=device, generator=torch.Generator(device).manual_seed(s)) < 0.5)
             .expand(count, sbs, sbs).contiguous() for s in range(2)]
    want = [_fresh(layer, blocks, attention_mask=m, sparsity_layout_mask=layer.layout) for m in masks]
    assert not torch.equal(want[0][0], want[1][0])
    for which in (0, 0, 0, 1, 1, 0, 1, 1, 1, 0, 0):
        _assert_same(_results(layer, blocks, attention_mask=masks[which], sparsity_layout_mask=layer.layout), want[which])
    layer.cache = {}
    plain = _fresh(layer, blocks)
    for which in (0, 0, None, 0, None):
        extra = {} if which is None else dict(attention_mask=masks[0], sparsity_layout_mask=layer.layout)
        _assert_same(_results(layer, blocks, **extra), plain if which is None else want[0])


def test_threads_that_share_a_cache(device):
    """Each on a stream of its own, with validation off: the way through the cache that looks nothing up again."""
    layer = _Layer(device, 32, False, n=9)
    blocks = [layer.inputs(torch.float16, 10 * t) for t in range(4)]
    want = [_results(layer, b) for b in blocks]
    torch.cuda.synchronize()
    failures = []

    def program(t):
        try:
            bs.utils.disable_validation()
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    _assert_same(_results(layer, blocks[t]), want[t])
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    threads = [threading.Thread(target=program, args=(t,)) for t in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    if failures:
        raise failures[0]

"""to_sparse of a layout that is used once: the host looks for the block count while the coordinates are enqueued."""

import pytest
import torch

import blksprs_amd as bs
from blksprs_amd import _capi
from blksprs_amd.utils import tools

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,density", [
    ((1, 1, 2), 1.0), ((1, 3, 5), 0.0), ((2, 9, 13), 0.4), ((1, 1, 2048), 0.5), ((3, 683, 1), 0.5), ((4, 64, 128), 0.1),
    ((8, 128, 128), 0.05),  # 2^17 entries: the last that takes this way
    ((1, 131, 1001), 0.02),  # beyond
])
def test_to_sparse_without_a_cache_counts_while_it_enqueues(device, shape, density):
    layout = (torch.rand(shape, generator=torch.Generator().manual_seed(sum(shape))) < density).to(device)
    assert tools.counts_while_enqueued(layout) == (layout.numel() <= 1 << 17)
    B, R, C = shape
    x = torch.randn((B, 16 * R, 16 * C), device=device)
    want = x.view(B, R, 16, C, 16).permute(0, 1, 3, 2, 4)[layout]
    for _ in range(3):
        assert torch.equal(torch.Tensor(bs.ops.to_sparse(x, layout, 16)), want)
    assert torch.equal(torch.Tensor(bs.ops.to_sparse(x, layout, 16, layout_cache={})), want)


def test_coordinates_of_a_layout_that_does_not_start_on_16_bytes(device):
    whole = torch.rand((1, 5000), device=device) < 0.3
    layout = whole.view(-1)[3:4995].view(2, 48, 52)
    coords, count = tools.nonzero_for_one_call(layout)
    assert count == int(layout.sum()) and torch.equal(coords, layout.nonzero()) and coords.is_contiguous()


def test_to_sparse_behind_queued_work_of_another_stream(device):
    stream = torch.cuda.Stream()
    x = torch.zeros((2, 256, 256), device=device)
    layout = torch.zeros((2, 16, 16), dtype=torch.bool, device=device)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(20_000_000)
        x.add_(1)
        layout[:, ::3, 1::2] = True
        out = bs.ops.to_sparse(x, layout, 16)
        n = out.size(0)
    stream.synchronize()
    assert n == 2 * 6 * 8 and bool((out == 1).all())


@pytest.mark.parametrize("entries,first", [(2048, 0), (1 << 17, 0), (5000, 3), ((1 << 21) + 2049, 0)])
def test_the_count_is_all_that_the_host_is_left(device, entries, first):
    """Counted from the layout, from the tiles' counts and by a scan of them: the host takes its word back as soon as it has seen
    the count, so nothing may be written beside it or after it."""
    whole = torch.rand(first + entries, device=device, generator=torch.Generator(device).manual_seed(entries)) < 0.3
    layout = whole[first:].view(torch.uint8)
    packed = torch.empty(entries, dtype=torch.int64, device=device)
    workspace = torch.empty(_capi.load().bsa_lut_workspace_bytes(entries), dtype=torch.uint8, device=device)
    words = torch.full((3,), 1 << 40, dtype=torch.int64, device="cpu").pin_memory()
    stream = _capi.stream(device)
    _capi.call("bsa_lut_packed_counted", layout.data_ptr(), entries, packed.data_ptr(), words[1:].data_ptr(), workspace.data_ptr(),
               workspace.numel(), stream)
    count = _capi.load().bsa_lut_counted_wait(words[1:].data_ptr(), stream)
    torch.cuda.synchronize()
    assert words.tolist() == [1 << 40, count, 1 << 40] and count == int(whole[first:].sum())
    expected = torch.where(layout != 0, layout.cumsum(0, dtype=torch.int64) - 1, -1)
    assert torch.equal(packed, expected)


def test_every_look_at_pinned_memory_is_a_counted_wait(device):
    """torch's own report of waits (sync debug mode) does not see them."""
    layout = torch.ones((1, 2, 2), dtype=torch.bool, device=device)
    x, cache = torch.zeros((1, 32, 32), device=device), {}
    full = torch.ones((1, 2, 1), dtype=torch.bool, device=device)
    blocks, attention_cache = torch.zeros((2, 16, 16), device=device), {}
    lengths = torch.tensor([32], device=device)

    def waits(call):
        before = _capi.host_waits
        call()
        return _capi.host_waits - before

    def attend():
        bs.ops.flash_attention(blocks, full, blocks, full, blocks, full, layout, 16, causal_lengths=lengths,
                               layout_cache=attention_cache)

    bs.ops.to_sparse(x, layout, 16, layout_cache=cache)
    assert [waits(lambda: bs.ops.to_sparse(x, layout, 16)) for _ in range(2)] == [1, 1]
    assert waits(lambda: bs.ops.to_sparse(x, layout, 16, layout_cache=cache)) == 0
    assert [waits(attend) for _ in range(2)] == [1, 0]  # the range of lengths that were seen before is known

"""The layout scan at the edges of its three ways to the sum in front of a tile (csrc/lut.hip: 2048 entries per tile; counted
again from the layout up to 2^17 aligned entries, from the tiles' counts up to 1024 tiles, by a scan of its own beyond)."""

import pytest
import torch

import blksprs_amd as bs
from blksprs_amd.utils import tools

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 2047, 2048, 2049, 4096 + 16, 2 ** 17 - 1, 2 ** 17, 2 ** 17 + 1, 2 ** 21, 2 ** 21 + 1])
@pytest.mark.parametrize("shift", [0, 1, 16])
@pytest.mark.parametrize("values", [(0, 1), (0, 128, 255)])
def test_scan(device, n, shift, values):
    g = torch.Generator(device=device).manual_seed(n + shift)
    choice = torch.tensor(values, dtype=torch.uint8, device=device)
    store = choice[torch.randint(0, len(values), (n + shift,), generator=g, device=device)]
    layout = store[shift:].view(1, 1, n)  # not 16-byte aligned for shift 1
    active = layout.reshape(-1) != 0
    before = active.long().cumsum(0) - active.long()
    info = tools.pack_layout(layout, row_len=n)
    assert torch.equal(info.packed, torch.where(active, before, -1))
    assert info.count == int(active.sum()) == info.max_per_row
    assert info.row_offsets.tolist() == [0, info.count]
    if n % 4 == 0:
        info = tools.pack_layout(layout, row_len=n // 4)
        assert info.row_offsets[:4].tolist() == before[::n // 4].tolist()
    assert torch.equal(tools.build_packed_indices(layout), torch.where(active, before, -1))


@pytest.mark.parametrize("build", ["to_dense", "softmax"])
def test_reverse_index_in_a_cache_is_complete(device, build):
    """A cache may be used on another stream right after the call that filled it: the host has waited for the scan, also
    behind a long queue on the stream."""
    from blksprs_amd.ops.conversion import to_dense_build_layout_cache
    from blksprs_amd.ops.softmax import softmax_build_layout_cache

    layout = torch.ones((2, 8, 8), dtype=torch.bool, device=device).tril()
    cold = {"to_dense": to_dense_build_layout_cache, "softmax": softmax_build_layout_cache}[build]
    cold({}, layout)  # loads what is loaded once
    big = torch.randn((4096, 4096), device=device)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(device=device)
    with torch.cuda.stream(side):
        for _ in range(8):
            big = (big @ big).clamp_(-1, 1)
        cold({}, layout)
        assert side.query()


def test_to_dense_without_a_cache_on_a_side_stream(device):
    layout = torch.ones((2, 8, 8), dtype=torch.bool, device=device).tril()
    x = torch.randn((int(layout.sum()), 32, 32), device=device)
    want = bs.ops.to_dense(x, layout, 32, layout_cache={})
    big = torch.randn((4096, 4096), device=device)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(device=device)
    with torch.cuda.stream(side):
        for _ in range(8):
            big = (big @ big).clamp_(-1, 1)
        late = x + big[0, 0] * 0
        got = bs.ops.to_dense(late, layout, 32)
    side.synchronize()
    assert torch.equal(got, want)

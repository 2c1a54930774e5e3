"""The layout scan at the edges of its three ways to the sum in front of a tile (csrc/lut.hip: 2048 entries per tile; counted
again from the layout up to 2^17 aligned entries, from the tiles' counts up to 1024 tiles, by a scan of its own beyond)."""

import pytest
import torch

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

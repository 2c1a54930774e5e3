"""Softmax of rows that several groups of lanes share: row lengths around the rounds of a group, rows that leave some groups
without a block in the last round, and rows much longer than the mean, whose lanes read them twice; and long rows that are not
shared, since the mean is short."""

import pytest
import torch

import blksprs_amd as bs
from oracle import blksprs_oracle as orc

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("sbs,lengths", [
    (16, range(1, 20)), (16, [1, 63, 64, 65, 127, 128, 129]), (16, [3] * 40 + [200]), (16, [260, 257, 300]),
    (32, range(14, 34)), (32, [40, 41, 64, 65, 72]), (64, [1, 2, 15, 16, 17, 18, 31, 32, 33]), (64, [64, 63, 66]),
    (128, [8, 15, 16, 17, 30, 33]), (256, [15, 16, 17, 31]), (512, [7, 8, 9]),
])
def test_softmax_of_rows_shared_by_groups_of_lanes(device, sbs, lengths):
    lengths = list(lengths)
    layout = torch.arange(max(lengths))[None, :] < torch.tensor(lengths)[:, None]
    layout = layout[:, torch.randperm(max(lengths), generator=torch.Generator().manual_seed(1))][None].contiguous()
    g = torch.Generator().manual_seed(sbs + len(lengths))
    n = sum(lengths)
    x, go = (torch.randn((n, sbs, sbs), generator=g) * s for s in (3.0, 1.0))
    x[0, 0, 0] = float("-inf")
    xd = x.to(device).requires_grad_(True)
    out = bs.ops.softmax(xd, layout.to(device), sbs)
    out.backward(go.to(device))
    y = orc.softmax(x.double(), layout.numpy(), sbs)
    # an exponential is off by the rounding of its argument (up to 32 / ln 2 in units of the last place of 16) and its own
    # two units, the sum and the quotient by a few more: 64 EPS of the value itself
    assert ((out.detach().double().cpu() - y).abs() <= 64 * EPS * y + 1e-37).all()
    # dx = y (g - s): s = sum y g is off by those 64 EPS and the additions of its terms, all below sum y |g| <= max |g| of a row
    dx = orc.softmax_backward(go.double(), y, layout.numpy(), sbs)
    assert ((xd.grad.double().cpu() - dx).abs() <= 256 * EPS * y * float(go.abs().max()) + 1e-37).all()


@pytest.mark.parametrize("sbs,blocks", [(16, 300), (16, 1200), (64, 300)])
@pytest.mark.parametrize("largest", [13.3, 15.7, 30.1])
def test_a_maximum_that_stays_through_a_long_row(device, sbs, blocks, largest):
    """A row of several hundred blocks among rows of one: its sum is carried through 38 to 150 chunks that bring no larger value."""
    layout = torch.zeros((1, 401, blocks), dtype=torch.bool)
    layout[0, 0] = layout[0, :, 0] = True
    x = torch.randn((blocks + 400, sbs, sbs), generator=torch.Generator().manual_seed(blocks))
    x[0, :, 0] = largest
    out = torch.Tensor(bs.ops.softmax(x.to(device), layout.to(device), sbs)).double().cpu()
    y = orc.softmax(x.double(), layout.numpy(), sbs)
    # as above: 64 EPS of an exponential and its sum, whose few hundred additions per lane are of positive terms
    assert ((out - y).abs() <= (64 + blocks / 4) * EPS * y + 1e-37).all()


@pytest.mark.parametrize("sbs", [16, 32, 64])
@pytest.mark.parametrize("long_rows", [[15, 16, 17], [24, 25, 31], [32, 33, 40], [8, 9, 65], [41, 47, 48, 49]])
def test_softmax_of_long_rows_among_short_ones(device, sbs, long_rows):
    """Means below 4.8 blocks: whole chunks of eight units, and ends of one to eight, in registers (up to 16 and 32) and beyond."""
    test_softmax_of_rows_shared_by_groups_of_lanes(device, sbs, [1, 2, 3] * 24 + long_rows)

"""fp32 products formed from bf16 parts (split_f32.h) over the exponents of their operands: no bit of a value is lost, whatever
the other operand makes of its size."""

import pytest
import torch

import blksprs_amd as bs
from tests.helpers import rand_blocks
from tests.test_split_f32_gpu import EPS, _compressed, _dense

pytestmark = pytest.mark.gpu


def _products(device, sbs, x, y, go):
    """O = x y, dX = go y^T, dY = x^T go of dense (1, ., .) operands, and the same in 64 bits."""
    ones = lambda t: torch.ones((1, t.shape[1] // sbs, t.shape[2] // sbs), dtype=torch.bool)
    lx, ly, lo = ones(x), ones(y), ones(go)
    xd, yd, gd = (_compressed(t, layout, sbs).contiguous().to(device) for t, layout in ((x, lx), (y, ly), (go, lo)))
    xd.requires_grad_(True), yd.requires_grad_(True)
    out = bs.ops.matmul(xd, lx.to(device), yd, ly.to(device), lo.to(device), sbs)
    got = (out, *torch.autograd.grad(out, (xd, yd), gd))
    x, y, go = x.double(), y.double(), go.double()
    want = (x @ y, go @ y.transpose(1, 2), x.transpose(1, 2) @ go)
    return [(name, _dense(g.detach().cpu(), layout, sbs), w, n) for name, g, layout, w, n in
            zip(("O", "dX", "dY"), got, (lo, lx, ly), want, (x.shape[2], y.shape[2], x.shape[1]))]


def _random(rows, cols, seed):
    return torch.randn((1, rows, cols), generator=torch.Generator().manual_seed(seed))


# Error against 64 bits, in the 2-norm, of sums of n products of random values.  Rounding a sum of n products of size 1 has an
# error of up to EPS sqrt(n) and a mean square of a third of that; 6 n / 16 roundings on the way up are worth 0.35 EPS sqrt(n) in
# all where sums grow like a random walk, and the instruction's own order of additions some of it.  Measured: 0.25.  With the two
# products of a third part left out the error is 58 EPS whatever n is, with one of them 41, without the product of the second
# parts 46 (in 64 bits).
def _bound(n):
    return 0.5 * EPS * max(n, 64) ** 0.5


@pytest.mark.parametrize("sbs", [64, 128])
@pytest.mark.parametrize("x_scale,y_scale", [(0, 0), (-115, 115), (-120, 120), (120, -120), (-118, 60), (-122, 40), (50, -121)])
def test_matmul_of_opposite_scales(device, sbs, x_scale, y_scale):
    x, y, go = (_random(*shape, seed) for seed, shape in enumerate(((2 * sbs, 3 * sbs), (3 * sbs, sbs), (2 * sbs, sbs))))
    for name, got, want, n in _products(device, sbs, x * 2.0 ** x_scale, y * 2.0 ** y_scale, go):
        assert float((got - want).norm() / want.norm()) < _bound(n), name


def test_matmul_of_rows_of_different_scales(device):
    """Rows of x and columns of y of their own scale each: every row and every column is as exact as it is alone."""
    sbs = 64
    rows = 2.0 ** torch.linspace(-120, 60, 2 * sbs).round()
    cols = 2.0 ** torch.linspace(40, -110, sbs).round()
    x, y, go = _random(2 * sbs, 3 * sbs, 1) * rows[:, None], _random(3 * sbs, sbs, 2) * cols, _random(2 * sbs, sbs, 3)
    sizes = (x.double().abs() @ y.double().abs(), go.double().abs() @ y.double().abs().transpose(1, 2),
             x.double().abs().transpose(1, 2) @ go.double().abs())
    # the mean square over every row and every column, against the sum of the sizes: 0.4 EPS where 192 products are of one size,
    # measured 0.36 to 0.73 over a tensor; without third parts from 8 EPS (products of one size) to 32.  2^-146: results that fp32
    # holds as subnormal numbers only
    for (name, got, want, n), size in zip(_products(device, sbs, x, y, go), sizes):
        error = ((got - want) / (EPS * size + 2.0 ** -146)).square()
        assert (error.mean(dim=1) < 4).all() and (error.mean(dim=2) < 4).all(), name


@pytest.mark.parametrize("sbs", [64, 128])
@pytest.mark.parametrize("lowest,highest", [(-126, -100), (-126, 100), (0, 0), (90, 127)])
def test_matmul_with_the_identity_is_exact(device, sbs, lowest, highest):
    """Every part of a value arrives: 24 random bits and exponents over the range, times one, come back bit for bit.  (0, 0): the
    third part alone, in values of 24 bits of which the first and the second part cancel in the sum with another value."""
    g = torch.Generator().manual_seed(sbs)
    side = 2 * sbs
    bits = torch.randint(2 ** 23, 2 ** 24, (1, side, side), generator=g).double() * (torch.randint(0, 2, (1, side, side), generator=g) * 2 - 1)
    eye = torch.eye(side)[None]
    if lowest == highest:
        top = (torch.round(bits / 2 ** 8) * 2 ** 8).float()  # 16 bits
        first = torch.stack((bits.float(), -top), dim=3).reshape(1, side, 2 * side)
        pick = torch.stack((eye, eye), dim=2).reshape(1, 2 * side, side)
        name, got, want, _ = _products(device, sbs, first, pick, eye)[0]
        assert torch.equal(got, want) and want.abs().max() <= 128
        return
    value = torch.ldexp(bits, torch.randint(lowest - 23, highest - 22, (1, side, side), generator=g)).float()
    other = torch.ldexp(bits.flip(1), torch.randint(lowest - 23, highest - 22, (1, side, side), generator=g)).float()
    for x, y, go, names in ((value, eye, other, ("O", "dX")), (eye, value, other, ("O", "dY"))):
        for name, got, want, _ in _products(device, sbs, x, y, go):
            if name in names:
                assert torch.equal(got, want), name


def _attention(device, sbs, nh, q, k, v, go, scale):
    n = q.shape[1] // sbs
    full = torch.ones((q.shape[0], n, nh), dtype=torch.bool)
    la = torch.ones((q.shape[0], n, n), dtype=torch.bool)
    ops = [_compressed(t, full, sbs).contiguous().to(device).requires_grad_(True) for t in (q, k, v)]
    fd = full.to(device)
    out = bs.ops.flash_attention(ops[0], fd, ops[1], fd, ops[2], fd, la.to(device), sbs, scale=scale)
    got = (out, *torch.autograd.grad(out, ops, _compressed(go, full, sbs).contiguous().to(device)))
    q, k, v, go = (t.double() for t in (q, k, v, go))
    p = torch.softmax(q @ k.transpose(1, 2) * scale, dim=-1)
    o = p @ v
    ds = p * (go @ v.transpose(1, 2) - (go * o).sum(-1, keepdim=True)) * scale
    want = (o, ds @ k, ds.transpose(1, 2) @ q, p.transpose(1, 2) @ go)
    return zip(("O", "dQ", "dK", "dV"), (_dense(g.detach().cpu(), full, sbs) for g in got), want)


@pytest.mark.parametrize("sbs,nh", [(32, 1), (32, 2), (32, 4), (64, 1), (64, 2)])
@pytest.mark.parametrize("exponents", [(-115, 115, 0, 0), (115, -115, 0, 0), (-123, 123, 0, 0), (0, 0, -118, 0), (0, 0, 0, -118),
                                       (0, 0, -118, 118), (0, 0, 118, -118), (60, -60, 60, -60), (-118, 20, 0, 0)])
def test_attention_of_opposite_scales(device, sbs, nh, exponents):
    """Relative errors (2-norm) against 64 bits, as for operands of size 1 (below 5e-7, tests/test_split_f32_gpu.py)."""
    rows, cols = 5 * sbs, nh * sbs
    q, k, v, go = (torch.randn((2, rows, cols), generator=torch.Generator().manual_seed(seed)) * 2.0 ** e
                   for seed, e in enumerate(exponents))
    for name, got, want in _attention(device, sbs, nh, q, k, v, go, cols ** -0.5):
        assert float((got - want).norm() / want.norm()) < 1e-6, name


@pytest.mark.parametrize("sbs,nh", [(32, 2), (32, 3), (64, 2)])
def test_attention_of_columns_of_different_scales(device, sbs, nh):
    """Columns of K, V, Q and dO of their own scales: every column of the result is as exact as it is alone.  The scores come from
    columns of size 1 (the other operand's are as large as this one's are small)."""
    rows, cols = 5 * sbs, nh * sbs
    q, k, v, go = (torch.randn((2, rows, cols), generator=torch.Generator().manual_seed(seed)) for seed in range(4))
    own = 2.0 ** torch.linspace(-118, 60, cols).round()
    for operands in ((q / own.clamp(2.0 ** -60, 2.0 ** 60), k * own, v, go), (q * own, k / own.clamp(2.0 ** -60, 2.0 ** 60), v, go),
                     (q, k, v * own.clamp(max=1), go), (q, k, v, go * own.clamp(max=1))):
        for name, got, want in _attention(device, sbs, nh, *operands, scale=cols ** -0.5):
            error, size = (got - want).norm(dim=1), want.norm(dim=1)
            assert (error <= 4e-6 * size).all(), (name, float((error / size).max()))

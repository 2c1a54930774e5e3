"""fp32 products formed from bf16 parts (split_f32.h): their error, values whose parts do not hold them (infinite, NaN, next to
the largest number), and the fp32 instruction that forms such sums again; values far below one."""

import pytest
import torch

import blksprs_amd as bs
from tests.helpers import rand_blocks, rand_layout

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _dense(blocks, layout, sbs):
    b, r, c = layout.shape
    out = torch.zeros((b, r, c, sbs, sbs), dtype=torch.float64)
    out[layout.nonzero(as_tuple=True)] = blocks.double()
    return out.permute(0, 1, 3, 2, 4).reshape(b, r * sbs, c * sbs)


def _compressed(dense, layout, sbs):
    b, r, c = layout.shape
    return dense.view(b, r, sbs, c, sbs).permute(0, 1, 3, 2, 4)[layout.nonzero(as_tuple=True)]


def _assert_like(got, want, bound, what):
    """Same infinities and NaN as ``want`` (64 bits, infinite from fp32's largest number on), elsewhere within ``bound``."""
    got, want = got.detach().double().cpu(), want.float().double()
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]), what
    assert ((got - want).abs() <= bound)[finite].all(), (what, float(((got - want).abs() / bound)[finite].max()))


def _matmul(device, sbs, R, K, C, density, change=None, x_scale=1.0, y_scale=1.0):
    B = 2
    lx, ly = rand_layout((B, R, K), density, 1, ensure_rows=True), rand_layout((B, K, C), density, 2, ensure_rows=True)
    lo = torch.ones((B, R, C), dtype=torch.bool)
    x, y = rand_blocks(int(lx.sum()), sbs, torch.float32, 3), rand_blocks(int(ly.sum()), sbs, torch.float32, 4)
    go = rand_blocks(int(lo.sum()), sbs, torch.float32, 5)
    x, y = x * x_scale, y * y_scale
    if change:
        change(x, y)
    xd, yd = (t.to(device).requires_grad_(True) for t in (x, y))
    out = bs.ops.matmul(xd, lx.to(device), yd, ly.to(device), lo.to(device), sbs)
    dx, dy = torch.autograd.grad(out, (xd, yd), go.to(device))
    x64, y64, g64 = _dense(x, lx, sbs), _dense(y, ly, sbs), _dense(go, lo, sbs)
    # pairs of blocks that are not there add nothing, where 0 * inf would add NaN: block by block over k
    o64 = torch.zeros_like(g64)
    dx64, dy64 = torch.zeros_like(x64), torch.zeros_like(y64)
    size_o, size_x, size_y = o64.clone(), dx64.clone(), dy64.clone()
    for b in range(B):
        for k in range(K):
            ks = slice(k * sbs, (k + 1) * sbs)
            for i in range(R):
                rows = slice(i * sbs, (i + 1) * sbs)
                for j in range(C):
                    cols = slice(j * sbs, (j + 1) * sbs)
                    if lx[b, i, k] and ly[b, k, j]:
                        o64[b, rows, cols] += x64[b, rows, ks] @ y64[b, ks, cols]
                        size_o[b, rows, cols] += x64[b, rows, ks].abs() @ y64[b, ks, cols].abs()
                    if ly[b, k, j]:
                        dx64[b, rows, ks] += g64[b, rows, cols] @ y64[b, ks, cols].T
                        size_x[b, rows, ks] += g64[b, rows, cols].abs() @ y64[b, ks, cols].T.abs()
                    if lx[b, i, k]:
                        dy64[b, ks, cols] += x64[b, rows, ks].T @ g64[b, rows, cols]
                        size_y[b, ks, cols] += x64[b, rows, ks].T.abs() @ g64[b, rows, cols].abs()
    for what, got, want, size, layout, n in (("O", out, o64, size_o, lo, K), ("dX", dx, dx64, size_x, lx, C), ("dY", dy, dy64, size_y, ly, R)):
        # six roundings for 16 values, three dropped products of up to EPS together, and what underflows.  A bound for the worst
        # case: tests/test_split_f32_range_gpu.py holds the mean square, which tells whether all six products are there
        roundings = 6 * n * sbs / 16 + 4
        bound = roundings * 2 * EPS * _compressed(size, layout, sbs) + 1e-37
        _assert_like(got, _compressed(want, layout, sbs), bound, what)


@pytest.mark.parametrize("sbs", [64, 128])
@pytest.mark.parametrize("R,K,C,density", [(1, 1, 1, 1.0), (3, 2, 5, 0.4), (1, 70, 2, 1.0)])
def test_matmul(device, sbs, R, K, C, density):
    _matmul(device, sbs, R, K if sbs == 64 else min(K, 34), C, density)


@pytest.mark.parametrize("x_scale,y_scale", [(2.0 ** -115, 1.0), (1.0, 2.0 ** -118), (2.0 ** 100, 2.0 ** 10), (2.0 ** -60, 2.0 ** -50)])
def test_matmul_of_small_and_large_operands(device, x_scale, y_scale):
    _matmul(device, 64, 2, 3, 2, 0.7, x_scale=x_scale, y_scale=y_scale)


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan"), 3.4e38])
def test_matmul_of_single_values(device, value):
    """One value of x and one of y; 3.4e38 rounds to infinity in bf16."""
    def change(x, y):
        if value == 3.4e38:
            x *= 2.0 ** -20
            y *= 2.0 ** -20
        x[0, 5, 40] = value
        y[-1, 63, 0] = value

    _matmul(device, 64, 2, 3, 2, 0.7, change)


def _attention(device, sbs, nh, change=None, grad_scale=1.0):
    B, n = 2, 5
    la, full = torch.ones((B, n, n), dtype=torch.bool), torch.ones((B, n, nh), dtype=torch.bool)
    q, k, v, go = (rand_blocks(B * n * nh, sbs, torch.float32, i) for i in range(4))
    go = go * grad_scale
    if change:
        change(q, k, v, go)
    ops = [t.to(device).requires_grad_(True) for t in (q, k, v)]
    fd = full.to(device)
    out = bs.ops.flash_attention(ops[0], fd, ops[1], fd, ops[2], fd, la.to(device), sbs)
    grads = torch.autograd.grad(out, ops, go.to(device))
    q, k, v, go = (_dense(t, full, sbs) for t in (q, k, v, go))
    scale = (nh * sbs) ** -0.5
    s = q @ k.transpose(1, 2) * scale
    p = torch.softmax(s, dim=-1)
    o = p @ v
    dv = p.transpose(1, 2) @ go
    ds = p * (go @ v.transpose(1, 2) - (go * o).sum(-1, keepdim=True)) * scale
    want = (o, ds @ k, ds.transpose(1, 2) @ q, dv)
    return (out, *grads), [_compressed(t, full, sbs) for t in want]


@pytest.mark.parametrize("sbs,nh", [(32, 1), (32, 2), (32, 3), (32, 4), (64, 1), (64, 2)])
@pytest.mark.parametrize("grad_scale", [1.0, 2.0 ** -112, 2.0 ** 100])
def test_attention(device, sbs, nh, grad_scale):
    """Relative errors (2-norm) against 64 bits; the largest seen is 4e-7."""
    got, want = _attention(device, sbs, nh, grad_scale=grad_scale)
    for what, g, w in zip(("O", "dQ", "dK", "dV"), got, want):
        g = g.detach().double().cpu()
        assert float((g - w).norm() / w.norm()) < 1e-6, what


@pytest.mark.parametrize("sbs,nh", [(32, 1), (32, 2), (32, 4), (64, 1), (64, 2)])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("where", ["v", "go"])
def test_attention_of_single_values(device, sbs, nh, value, where):
    """A value of V or of dO that its parts do not hold: what it reaches is what it is in 64 bits, the rest as exact as ever."""
    def change(q, k, v, go):
        (v if where == "v" else go)[3, 7, 11] = value

    got, want = _attention(device, sbs, nh, change)
    names = ("O", "dQ", "dK", "dV")
    for what, g, w in zip(names, got, want):
        g = g.detach().double().cpu()
        if where == "go" and what in ("O", "dV") or where == "v" and what in ("O", "dV"):
            _assert_like(g, w, 1e-4 + 1e-4 * w.abs(), what)
        elif value != 3.4e38:
            assert not torch.isfinite(g).all(), what
            untouched = torch.isfinite(w)
            assert torch.isfinite(g[untouched]).all(), what


@pytest.mark.parametrize("sbs,nh", [(32, 2), (64, 1)])
def test_attention_of_infinite_keys(device, sbs, nh):
    """Scores of +inf make NaN of a query's row, scores of -inf leave a key out."""
    def change(q, k, v, go):
        k[2, 1, 3] = float("inf")

    got, want = _attention(device, sbs, nh, change)
    _assert_like(got[0], want[0], 1e-4 + 1e-4 * want[0].abs(), "O")

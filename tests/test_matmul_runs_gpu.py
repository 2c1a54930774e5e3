"""The matmul kernels for blocks of 16 and 32 (csrc/matmul.hip: matmul_runs32_kernel, matmul_small16_kernel,
matmul_small16_f32_kernel) where they can go wrong: output blocks without a pair in front of, between and behind others, lists
longer than the 64 entries of a window, launches of one, two and more output blocks per wave."""

import importlib

import pytest
import torch

import blksprs_amd as bs

mm = importlib.import_module("blksprs_amd.ops.matmul")

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _dense(blocks, layout, sbs):
    B, R, C = layout.shape
    out = torch.zeros((B, R, C, sbs, sbs), dtype=torch.float64, device=blocks.device)
    out[layout] = blocks.detach().double()
    return out.transpose(2, 3).reshape(B, R * sbs, C * sbs)


def _blocks(dense, layout, sbs):
    B, R, C = layout.shape
    return dense.reshape(B, R, sbs, C, sbs).transpose(2, 3)[layout]


def _check(got, want, magnitude, terms, dtype):
    # fp32 sums of `terms` products in any order, rounded once to the operand type: their magnitude is what the absolute
    # values add up to
    bound = magnitude * (terms * EPS[torch.float32]) + want.abs() * EPS[dtype] * 1.01 + 1e-30
    assert got.dtype == dtype and bool(((got.double() - want).abs() <= bound).all())


def _run(device, dtype, sbs, lx, ly, lo, seed):
    g = torch.Generator(device=device).manual_seed(seed)
    rand = lambda layout: torch.randn((int(layout.sum()), sbs, sbs), generator=g, device=device).to(dtype)
    x, y, grad = rand(lx).requires_grad_(), rand(ly).requires_grad_(), rand(lo)
    out = bs.ops.matmul(x, lx, y, ly, lo, sbs)
    dx, dy = torch.autograd.grad(out, (x, y), grad)
    X, Y, G = _dense(x, lx, sbs), _dense(y, ly, sbs), _dense(grad, lo, sbs)
    for got, a, b, layout in ((out, X, Y, lo), (dx, G, Y.mT.contiguous(), lx), (dy, X.mT.contiguous(), G, ly)):
        want = _blocks(torch.bmm(a, b), layout, sbs)
        magnitude = _blocks(torch.bmm(a.abs(), b.abs()), layout, sbs)
        _check(got.detach(), want, magnitude, a.size(2), dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sbs", [16, 32])
@pytest.mark.parametrize("B,R,K,C,density", [(1, 1, 1, 1, 1.0), (2, 3, 5, 4, 0.3), (1, 2, 70, 3, 1.0), (1, 3, 130, 2, 0.6),
                                             (3, 9, 8, 11, 0.1)])
def test_lists(device, dtype, sbs, B, R, K, C, density):
    g = torch.Generator().manual_seed(R * K * C)
    lx, ly, lo = (torch.rand(shape, generator=g) < density for shape in ((B, R, K), (B, K, C), (B, R, C)))
    lo = lo | (torch.rand((B, R, C), generator=g) < 0.5)  # many blocks without a pair
    for layout in (lx, ly, lo):
        layout[0, 0, 0] = True
    _run(device, dtype, sbs, lx.to(device), ly.to(device), lo.to(device), seed=K)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sbs,B,n", [(16, 17, 62), (16, 26, 62), (32, 2, 79), (32, 5, 71), (32, 7, 76)])
def test_runs(device, dtype, sbs, B, n):
    """65348 and 99944 output blocks of 16 (one and three per wave), 12482, 25205 and 40432 of 32 (one, two and three)."""
    g = torch.Generator().manual_seed(n)
    lx, ly = torch.rand((B, n, 3), generator=g) < 0.5, torch.rand((B, 3, n), generator=g) < 0.5
    lx[0, 0, 0] = ly[0, 0, 0] = True
    _run(device, dtype, sbs, lx.to(device), ly.to(device), torch.ones((B, n, n), dtype=torch.bool, device=device), seed=n)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,R,K,C,density", [(1, 1, 12, 1, 1.0), (2, 17, 40, 33, 0.6), (1, 5, 70, 19, 1.0), (3, 16, 24, 16, 0.75)])
def test_order_of_blocks(device, dtype, B, R, K, C, density):
    """Products of 12 and more pairs per output block follow the work order (super-tiles that are not whole, counts that
    are no multiple of a workgroup's four blocks); any order, or none, gives the same bits."""
    sbs, g = 32, torch.Generator().manual_seed(R * K * C)
    lx, ly = torch.rand((B, R, K), generator=g) < density, torch.rand((B, K, C), generator=g) < density
    lo = torch.ones((B, R, C), dtype=torch.bool)
    lx, ly, lo = lx.to(device), ly.to(device), lo.to(device)
    _run(device, dtype, sbs, lx, ly, lo, seed=C)
    cache = {}
    gd = torch.Generator(device=device).manual_seed(C)
    x, y = (torch.randn((int(layout.sum()), sbs, sbs), generator=gd, device=device).to(dtype) for layout in (lx, ly))
    out = bs.ops.matmul(x, lx, y, ly, lo, sbs, layout_cache=cache)
    plan = cache["plan"]
    assert mm._follows_order(plan.pairs.numel() // 2, plan.n_out, sbs)
    for order in (None, torch.randperm(plan.n_out, generator=gd, device=device).to(torch.int32)):
        other = mm._launch(x, y, plan.pair_offsets, plan.pairs, order, plan.n_out, sbs, False, False)
        assert torch.equal(other, out)

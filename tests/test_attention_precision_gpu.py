"""Rounding of the attention kernels for blocks of 16 and 32: probabilities are rounded against the exact running maximum
of their row, and the score a maximum or lse comes from differs from it by exactly zero."""

import math

import pytest
import torch

import blksprs_amd as bs
from tests.helpers import rand_blocks

pytestmark = pytest.mark.gpu


def _dense(blocks, batches, sbs):
    """Full layouts: [batches * rows * slices, sbs, sbs] -> [batches, rows * sbs, slices * sbs]."""
    slices = 64 // sbs
    t = blocks.double().view(batches, -1, slices, sbs, sbs)
    return t.permute(0, 1, 3, 2, 4).reshape(batches, -1, 64)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sbs", [16, 32])
@pytest.mark.parametrize("n_keys,batches,scale", [(1024, 4, 1 / 8), (1024, 4, 3 / 4), (256, 80, 1 / 8), (512, 140, 1 / 8)])
def test_probabilities_are_rounded_against_the_exact_maximum(device, dtype, sbs, n_keys, batches, scale):
    """Error against 64 bits, next to that of the same arithmetic on dense tensors: probabilities relative to the row's
    maximum, rounded to the operand type, products in 64 bits, one rounding of the output.  A kernel that follows the
    maximum key block by key block rounds some probabilities relative to an earlier one, in either direction; over 2 x 10^4
    rows that is below 3 % (the dense arithmetic relative to the maximum of the first half of the keys differs by 2 %).
    A reference that may lie up to 2^8 below the maximum is 8 to 10 % further off.  Launches with four, two and one wave
    per query block."""
    n_queries, slices = (1024 if batches == 4 else 512), 64 // sbs
    q, k, v = (rand_blocks(batches * n * slices // sbs, sbs, dtype, seed).to(device)
               for n, seed in ((n_queries, 1), (n_keys, 2), (n_keys, 3)))
    layout = lambda rows, cols: torch.ones((batches, rows // sbs, cols // sbs), dtype=torch.bool, device=device)
    lq, lk = layout(n_queries, 64), layout(n_keys, 64)
    out = bs.ops.flash_attention(q, lq, k, lk, v, lk, layout(n_queries, n_keys), sbs, scale=scale)
    got, exact_error, dense_error, norm = _dense(out, batches, sbs), 0.0, 0.0, 0.0
    q, k, v = (_dense(t, batches, sbs) for t in (q, k, v))
    for b in range(batches):
        s = (q[b] @ k[b].T.contiguous()) * scale
        p = torch.exp(s - s.max(dim=1, keepdim=True).values)
        total = p.sum(dim=1, keepdim=True)
        want = p @ v[b] / total
        rounded = (p.to(dtype).double() @ v[b] / total).to(dtype).double()
        exact_error += float((got[b] - want).square().sum())
        dense_error += float((rounded - want).square().sum())
        norm += float(want.square().sum())
    assert math.sqrt(exact_error / norm) <= 1.03 * math.sqrt(dense_error / norm), (
        math.sqrt(exact_error / norm), math.sqrt(dense_error / norm))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sbs", [16, 32])
def test_a_query_that_sees_one_key_returns_its_value(device, dtype, sbs):
    """Its probability is exactly one, forward and backward: O is V of that key, and its dO arrives in dV as it is."""
    n, slices = 3, 64 // sbs
    lay = torch.ones((1, n, slices), dtype=torch.bool, device=device)
    la = torch.eye(n, dtype=torch.bool, device=device)[None].contiguous()
    q, k, v, go = (rand_blocks(n * slices, sbs, dtype, seed, 3.0).to(device) for seed in range(4))
    # key i alone is left of each block for query i
    mask = ~torch.eye(sbs, dtype=torch.bool, device=device).expand(n, sbs, sbs).contiguous()
    for t in (q, k, v):
        t.requires_grad_(True)
    out = bs.ops.flash_attention(q, lay, k, lay, v, lay, la, sbs, scale=0.37, attention_mask=mask, sparsity_layout_mask=la)
    dv, = torch.autograd.grad(out, v, go)
    assert torch.equal(out.detach(), v.detach())
    assert torch.equal(dv, go)


@pytest.mark.parametrize("sbs", [16, 32])
@pytest.mark.parametrize("causal", [False, True])
def test_fp32_sums_do_not_depend_on_the_number_of_rows(device, sbs, causal):
    """fp32 sums of a row are formed in four parts whatever the launch: a batch entry's output and gradients are the
    same bits alone (few rows) and among 140 or 300 others (thousands of rows)."""
    n, slices = 32, 64 // sbs
    la = torch.ones((1, n, n), dtype=torch.bool, device=device)
    if causal:
        la = la.tril().contiguous()
    lay = torch.ones((1, n, slices), dtype=torch.bool, device=device)
    alone = [rand_blocks(n * slices, sbs, torch.float32, seed).to(device) for seed in range(4)]

    def step(batches):
        q, k, v, go = (t.repeat(batches, 1, 1) for t in alone)
        for t in (q, k, v):
            t.requires_grad_(True)
        full, layout = (t.expand(batches, -1, -1).contiguous() for t in (lay, la))
        out = bs.ops.flash_attention(q, full, k, full, v, full, layout, sbs)
        return (out.detach(), *torch.autograd.grad(out, (q, k, v), go))

    first = step(1)
    for batches in (140, 300):
        for name, got, want in zip(("O", "dQ", "dK", "dV"), step(batches), first):
            assert torch.equal(got, want.repeat(batches, 1, 1)), (name, batches)

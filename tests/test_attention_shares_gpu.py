"""Uneven attention layouts: rows shared by as many waves as their lists are long (attn_shares.hip, and the kernels of
attn_small_fwd.hip and attn_small_bwd.hip that read the shares)."""

import ctypes

import pytest
import torch

import blksprs_amd as bs
from blksprs_amd import _capi
from oracle import blksprs_oracle as orc
from tests.test_attention_gpu import TOL, assert_close, rand_blocks

pytestmark = pytest.mark.gpu


def _parts(n, piece, least, sbs, dtype):
    most = max(6 * piece, 4 * (piece + (6 if dtype == torch.float32 else 24) * (2 if sbs == 16 else 1)))
    parts = 1 if 2 * n <= 3 * piece else 2 if n <= 3 * piece else 4 if n <= most else 4 * -(-n // (4 * piece))
    return max(parts, least)


@pytest.mark.parametrize("B,rows", [(1, 1), (1, 70), (3, 9), (8, 8), (11, 130), (17, 300), (300, 3)])
@pytest.mark.parametrize("sbs,dtype", [(16, torch.bfloat16), (64, torch.float32)])
@pytest.mark.parametrize("piece", [1, 5, 40])
def test_every_part_of_every_row_is_handed_out_once(device, B, rows, sbs, dtype, piece):
    g = torch.Generator().manual_seed(B + rows + piece)
    lengths = torch.randint(0, 12, (B * rows,), generator=g)
    lengths[torch.rand(B * rows, generator=g) < 0.1] = 400
    offsets = torch.cat([torch.zeros(1, dtype=torch.long), lengths.cumsum(0)]).int().to(device)
    halves = 2 if sbs == 64 else 1
    a = _capi.AttnArgs()
    a.B, a.nq, a.nk, a.nh, a.nhv, a.sbs, a.dtype = B, 5, rows, 1, 1, sbs, _capi.DTYPE_CODES[dtype]
    a.query_offsets = offsets.data_ptr()
    # what every row gets without shares: fp32 four waves, 16-bit by the number of rows; never more than a list has steps
    steps = -(-halves * 5 // (2 if sbs == 16 else 1))
    wanted = 4 if dtype == torch.float32 or B * rows <= 512 else 2
    least = min(wanted, 4 if steps >= 3 else steps)
    entries = halves * int(lengths.sum())
    max_groups = 8 * (-(-rows // 8) * (B // 8 * min(rows, 8) + B % 8) + entries // (4 * piece) + 1)
    max_merges = entries // (6 * piece) + 1
    groups = torch.full((max_groups + 1, _capi.SHARE_INTS), -7, dtype=torch.int32, device=device)
    merges = torch.full((max_merges + 1, 4), -7, dtype=torch.int32, device=device)
    stats = torch.zeros(3, dtype=torch.int64, device=device)
    _capi.call("bsa_attn_shares_build", ctypes.byref(a), 1, piece, max_groups, max_merges, groups.data_ptr(), merges.data_ptr(),
               stats.data_ptr(), _capi.stream(torch.device("cuda", torch.cuda.current_device())))
    per_xcd, n_merges, n_slots = stats.tolist()
    assert (groups[max_groups] == -7).all() and (merges[max_merges] == -7).all()
    assert 8 * per_xcd <= max_groups and n_merges <= max_merges
    seen, slots = {}, {}
    for j, (o0, o1, o2, o3, b0, b1, b2, b3, first, parts, slot, _) in enumerate(groups[:max_groups].tolist()):
        waves = min(parts, 4)
        owners = list(zip((b0, b1, b2, b3), (o0, o1, o2, o3)))
        for w, (b, own) in enumerate(owners):
            assert owners[w // waves * waves] == (b, own)  # the waves of a row are neighbours
            if own < 0:
                continue
            assert j < 8 * per_xcd
            seen.setdefault((b, own), []).append((first + w % waves, parts))
            if slot >= 0:
                assert slots.setdefault(slot, (b, own, first)) == (b, own, first)
    assert len(seen) == B * rows and sorted(slots) == list(range(n_slots))
    for (b, own), got in seen.items():
        want = _parts(halves * int(lengths[b * rows + own]), piece, least, sbs, dtype)
        assert sorted(got) == [(p, want) for p in range(want)]
    merged = {(b, own): (slot, n) for b, own, slot, n in merges[:n_merges].tolist()}
    assert len(merged) == n_merges and set(merged) == {key for key, got in seen.items() if got[0][1] > 4}
    for key, (slot, n) in merged.items():
        assert 4 * n == seen[key][0][1]
        assert [slots[slot + i] for i in range(n)] == [(*key, 4 * i) for i in range(n)]


def _run(device, dtype, sbs, layout, nh, seed, use_mask, use_bias, use_causal, expect):
    B, nq, nk = layout.shape
    g = torch.Generator().manual_seed(seed)
    full = lambda rows: torch.ones((B, rows, nh), dtype=torch.bool)
    q, k, v = (rand_blocks(B * rows * nh, sbs, dtype, seed + i) for i, rows in enumerate((nq, nk, nk)))
    mask = lmask = bias = lbias = lengths = None
    if use_mask:
        lmask = layout & orc.random_layout(tuple(layout.shape), 0.5, g)
        mask = torch.rand((int(lmask.sum()), sbs, sbs), generator=g) < 0.3
    if use_bias:
        lbias = layout & orc.random_layout(tuple(layout.shape), 0.5, g)
        bias = rand_blocks(int(lbias.sum()), sbs, dtype, seed + 4)
    if use_causal:
        lengths = torch.randint(1, nq * sbs + 1, (B,), generator=g)
    to = lambda t: None if t is None else t.to(device)
    ops = [t.to(device).requires_grad_(True) for t in (q, k, v)] + ([bias.to(device).requires_grad_(True)] if use_bias else [])
    cache = {}
    out = bs.ops.flash_attention(ops[0], to(full(nq)), ops[1], to(full(nk)), ops[2], to(full(nk)), to(layout), sbs,
                                 attention_mask=to(mask), sparsity_layout_mask=to(lmask), causal_lengths=to(lengths),
                                 attention_bias=ops[3] if use_bias else None, sparsity_layout_bias=to(lbias), layout_cache=cache)
    shares = cache["tables"].shares[(sbs, dtype, True)]
    assert [side is not None for side in shares] == [expect, expect]
    if expect:
        assert all(side.n_merges > 0 for side in shares)
    refs = [t.double().requires_grad_(True) for t in (q, k, v)] + ([bias.double().requires_grad_(True)] if use_bias else [])
    ref = orc.flash_attention(refs[0], full(nq).numpy(), refs[1], full(nk).numpy(), refs[2], full(nk).numpy(), layout.numpy(), sbs,
                              mask=mask, layout_mask=None if lmask is None else lmask.numpy(),
                              bias=refs[3] if use_bias else None, layout_bias=None if lbias is None else lbias.numpy(),
                              causal_lengths=lengths, acc_dtype=torch.float64)
    go = rand_blocks(out.size(0), sbs, dtype, seed + 5)
    out.backward(go.to(device))
    ref.backward(go.double())
    for name, got, want in zip(("O", "dQ", "dK", "dV", "dBias"), (out, *(t.grad for t in ops)), (ref, *(t.grad for t in refs))):
        # dBias = P (dP - delta), elementwise: delta sums head_dim products of dO with O rounded to the operand type, whose errors
        # are up to u = eps / 2 and about 0.4 u in the mean square: 2 u sqrt(head_dim) is five standard deviations where P is 1
        rounding = torch.finfo(dtype).eps * (nh * sbs) ** 0.5 if name == "dBias" and dtype != torch.float32 else 0.0
        assert_close(got, want, TOL[dtype] + rounding, name)


@pytest.mark.parametrize("dtype,sbs,nh", [(torch.float16, 16, 1), (torch.bfloat16, 16, 5), (torch.float32, 16, 3),
                                          (torch.bfloat16, 32, 2), (torch.float16, 32, 3), (torch.float32, 32, 1),
                                          (torch.float32, 64, 1)])
@pytest.mark.parametrize("use_mask,use_bias,use_causal", [(False, False, False), (True, True, False), (True, True, True)])
def test_long_rows_among_short_ones(device, dtype, sbs, nh, use_mask, use_bias, use_causal):
    """Global rows and columns among rows of one, two and ten blocks and empty ones: rows of one wave, two, four and of several
    workgroups in one launch."""
    n = 250 if sbs == 16 else 68 if sbs == 64 else 128
    layout = torch.zeros((2, n, n), dtype=torch.bool)
    layout[:, :2] = True
    layout[:, :, n // 2] = True
    layout[0, :, 3] = True
    i = torch.arange(n)
    layout |= (i[:, None] - i[None, :]).abs() <= (i % 6 == 0).long()[:, None] * 5
    layout[1, 7] = False
    _run(device, dtype, sbs, layout, nh, seed=sbs + nh, use_mask=use_mask, use_bias=use_bias, use_causal=use_causal, expect=True)


def test_even_layouts_go_without(device):
    _run(device, torch.bfloat16, 32, torch.ones((2, 20, 20), dtype=torch.bool), 2, seed=1, use_mask=False, use_bias=False,
         use_causal=False, expect=False)


def test_capture_without_and_with_kept_shares(device):
    """Under capture nothing is built; a cache that holds the shares replays with them, on new values, like an eager call."""
    n, sbs = 260, 16
    layout = torch.eye(n, dtype=torch.bool, device=device)[None].repeat(2, 1, 1)
    layout[:, 0] = True
    full = torch.ones((2, n, 2), dtype=torch.bool, device=device)
    make = lambda seed: [rand_blocks(2 * n * 2, sbs, torch.bfloat16, seed + i).to(device) for i in range(3)]
    call = lambda ops, cache: bs.ops.flash_attention(ops[0], full, ops[1], full, ops[2], full, layout, sbs, layout_cache=cache)
    for kept in (False, True):
        cache, static = {}, make(1)
        call(static, cache)
        assert cache["tables"].shares[(sbs, torch.bfloat16, False)][0].n_merges == 2
        if not kept:
            cache["tables"].shares.clear()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        bs.utils.disable_validation()  # its checks read the device
        try:
            with torch.cuda.graph(graph):
                out = call(static, cache)
        finally:
            bs.utils.enable_validation()
        assert bool(cache["tables"].shares) == kept
        for seed in (10, 20, 30):
            fresh = make(seed)
            for s, f in zip(static, fresh):
                s.copy_(f)
            graph.replay()
            torch.cuda.synchronize()
            assert_close(out, call(fresh, {}), 2e-2, f"replay {seed}")

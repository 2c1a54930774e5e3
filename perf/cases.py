"""The work that is timed: block-sparse attention, matrix products, softmax and conversion as a program calls them.

A case is a dict of plain values, ``op`` naming the path:

``attention``  ``bs.ops.flash_attention`` on compressed Q, K and V with the layout metadata kept in a cache, forward
               (``train`` false: inference) or forward and backward.  ``pattern``: ``bernoulli`` (every block with
               probability ``density``), ``bigbird`` (window of four blocks either side, two global block rows and
               columns, three random blocks per row, a causal mask tensor inside the layout), ``causal`` (all of the
               lower triangle, padded sequences, the native predicate of ``causal_lengths``) or ``window`` (causal
               attention to the last ``window`` tokens of padded sequences, the compact mask of the library's own
               builder).
``matmul``     ``bs.ops.matmul`` of two layouts of ``density`` with their product layout as output, forward or
               forward and both gradients.
``softmax``    ``bs.ops.softmax``, block-causal layout plus ``density`` of the blocks above the diagonal, forward or
               forward and backward.
``convert``    a dense tensor whose blocks are mostly zero: its layout is found, it is compressed and expanded again,
               without caches, since a program that does this has a new layout every time.

Ranges: 16-bit and fp32 operands (softmax: fp32 only, as the operator), block sizes 16, 32, 64 (matmul, softmax and
conversion also 128), head dimensions 32 to 128, sequences of 256 to 8192 tokens, matrices of 256 to 4096 a side, any
number of blocks per side and batch entries between.  Argument validation is off, as in a program past its first
steps (with it on, every call waits for the device several times).
"""

import functools
import math

import torch

import blksprs_amd as bs

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # the smallest attention call of a program: one short prompt, a few heads; latency and launches
        dict(name="attention_small", op="attention", dtype="bf16", sbs=32, heads=8, seq=256, head_dim=64,
             pattern="causal", train=False),
        # the reference's own attention benchmark (fp32, sbs 32, half of the blocks), as a training step
        dict(name="attention_fp32_train", op="attention", dtype="fp32", sbs=32, heads=8, seq=2048, head_dim=64,
             pattern="bernoulli", density=0.5, train=True),
        # long-context training: BigBird layout at block size 64, explicit causal mask
        dict(name="attention_long_train", op="attention", dtype="bf16", sbs=64, heads=64, seq=8192, head_dim=128,
             pattern="bigbird", train=True),
        # mixed-precision training of local causal attention on padded sequences at block size 32
        dict(name="attention_window_train", op="attention", dtype="fp16", sbs=32, heads=48, seq=4096, head_dim=64,
             pattern="window", window=1024, train=True),
        # prefill of padded prompts at the finest block size; 129 blocks, so nothing divides evenly
        dict(name="attention_prefill", op="attention", dtype="bf16", sbs=16, heads=32, seq=2064, head_dim=64,
             pattern="causal", train=False),
        # the smallest product: two batch entries of 256 x 256, latency of one call
        dict(name="matmul_small", op="matmul", dtype="fp32", sbs=32, batch=2, m=256, k=256, n=256, density=0.5,
             train=False),
        # a large 16-bit product with both gradients at block size 64
        dict(name="matmul_train", op="matmul", dtype="bf16", sbs=64, batch=16, m=4096, k=4096, n=4096, density=0.25,
             train=True),
        # a 16-bit product with both gradients at block size 32, no side a multiple of a larger tile
        dict(name="matmul_sbs32_train", op="matmul", dtype="bf16", sbs=32, batch=8, m=2976, k=4064, n=2080,
             density=0.25, train=True),
        # very sparse, very small blocks: gathers and lookup tables count more than products
        dict(name="matmul_sbs16_train", op="matmul", dtype="fp16", sbs=16, batch=64, m=2048, k=2048, n=2048,
             density=0.05, train=True),
        # a full-precision product with both gradients
        dict(name="matmul_fp32_train", op="matmul", dtype="fp32", sbs=64, batch=8, m=2048, k=2048, n=2048,
             density=0.25, train=True),
        # attention probabilities of the unfused path: fp32 softmax with its gradient
        dict(name="softmax_train", op="softmax", dtype="fp32", sbs=64, batch=32, n=2048, density=0.1, train=True),
        # compressing and expanding a large 16-bit tensor whose layout is not known beforehand
        dict(name="convert", op="convert", dtype="bf16", sbs=64, batch=16, m=4096, n=4096, density=0.25),
    ]


# ---------------------------------------------------------------------------------------------------- drawn cases

def _spread(rng, low, high):
    """A whole number between ``low`` and ``high``, spread over their logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _drawn_attention(rng):
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp16", "fp32"])
    sbs = rng.choice([16, 32, 64])
    # head dimensions in whole blocks, up to 128
    head_dim = sbs * rng.randint(1 if sbs > 16 else 2, 128 // sbs)
    case = dict(op="attention", dtype=dtype, sbs=sbs, head_dim=head_dim,
                pattern=rng.choice(["bernoulli", "bigbird", "causal", "window"]), train=rng.random() < 0.5)
    if case["pattern"] == "bernoulli":
        case["density"] = round(rng.uniform(0.1, 0.6), 3)
    if case["pattern"] == "window":
        case["window"] = _spread(rng, 128, 1024)
    case["seq"] = sbs * _spread(rng, 256 // sbs, (8192 if sbs == 64 else 4096) // sbs)
    case["heads"] = _spread(rng, 1, 64)
    # smaller blocks, wider operands and many head slices cost more for the same arithmetic
    limit = 5e10
    if head_dim // sbs > 4:
        limit = 8e8
    elif dtype == "fp32" or sbs == 16:
        limit = 1e10
    while work(case)["flops"] > limit:
        if case["heads"] > 1:
            case["heads"] = (case["heads"] + 1) // 2
        else:
            case["seq"] = sbs * max(case["seq"] // sbs * 2 // 3, 1)
    return case


def _drawn_matmul(rng):
    dtype = rng.choice(["bf16", "fp16", "fp32"])
    sbs = rng.choice([16, 32, 64, 128])
    sides = {side: sbs * _spread(rng, max(256 // sbs, 2), 4096 // sbs) for side in ("m", "k", "n")}
    case = dict(op="matmul", dtype=dtype, sbs=sbs, batch=_spread(rng, 1, 16), **sides,
                density=round(rng.uniform(0.05, 0.4) * (0.5 if sbs == 16 else 1.0), 3), train=rng.random() < 0.5)
    limit = 2e9 if sbs == 16 else 3e10 if dtype == "fp32" else 1e11
    while work(case)["flops"] > limit:
        if case["batch"] > 1:
            case["batch"] = (case["batch"] + 1) // 2
        else:
            longest = max(("m", "k", "n"), key=lambda side: case[side])
            case[longest] = sbs * max(case[longest] // sbs * 2 // 3, 1)
    return case


def draw(rng):
    op = rng.choices(["attention", "matmul", "softmax", "convert"], [5, 4, 1, 1])[0]
    if op == "attention":
        return _drawn_attention(rng)
    if op == "matmul":
        return _drawn_matmul(rng)
    sbs = rng.choice([16, 32, 64, 128])
    if op == "softmax":
        return dict(op="softmax", dtype="fp32", sbs=sbs, batch=_spread(rng, 1, 32),
                    n=sbs * _spread(rng, 256 // sbs, 2048 // sbs), density=round(rng.uniform(0.0, 0.3), 3),
                    train=rng.random() < 0.5)
    return dict(op="convert", dtype=rng.choice(["bf16", "fp16", "fp32"]), sbs=sbs, batch=_spread(rng, 1, 8),
                m=sbs * _spread(rng, 256 // sbs, 4096 // sbs), n=sbs * _spread(rng, 256 // sbs, 4096 // sbs),
                density=round(rng.uniform(0.05, 0.6), 3))


# ---------------------------------------------------------------------------------------------------- inputs

def _bernoulli(shape, density, number):
    """Every block with probability ``density``, at least one per row.  Drawn from ``number``, not from a case's seed:
    another seed shuffles rows and columns, so that the counts of blocks and of block pairs stay what they are."""
    g = torch.Generator(device="cuda").manual_seed(number)
    layout = torch.rand(shape, generator=g, device="cuda") < density
    columns = torch.randint(0, shape[2], (*shape[:2], 1), generator=g, device="cuda")
    first = torch.zeros_like(layout).scatter_(2, columns, True)
    return layout | (first & ~layout.any(dim=2, keepdim=True))


def _shuffled(count, g):
    return torch.randperm(count, generator=g, device="cuda")


def _bigbird(heads, n, g):
    i = torch.arange(n, device=g.device)
    rows, cols = i[:, None], i[None, :]
    fixed = ((rows - cols).abs() <= 4) | (rows < 2) | (cols < 2)
    chosen = torch.rand((heads, n, n), generator=g, device=g.device).argsort(dim=-1)[..., :3]
    return torch.zeros((heads, n, n), dtype=torch.bool, device=g.device).scatter_(2, chosen, True) | fixed


def _sequence_lengths(case, g):
    """Padded batches: between half and all of the positions are in use, evenly spread, in any order."""
    lengths = torch.linspace(case["seq"], case["seq"] // 2, case["heads"], device="cuda").long()
    return lengths[_shuffled(case["heads"], g)].contiguous()


def _attention_pattern(case, g):
    """(attention layout, keyword arguments of flash_attention that go with it)"""
    heads, sbs = case["heads"], case["sbs"]
    n = case["seq"] // sbs
    if case["pattern"] == "bernoulli":
        layout = _bernoulli((heads, n, n), case["density"], 1)
        return layout[:, _shuffled(n, g)][:, :, _shuffled(n, g)].contiguous(), {}
    if case["pattern"] == "causal":
        layout = torch.ones((n, n), dtype=torch.bool, device=g.device).tril().expand(heads, n, n).contiguous()
        return layout, dict(causal_lengths=_sequence_lengths(case, g))
    if case["pattern"] == "window":
        lengths = _sequence_lengths(case, g)
        layout = bs.layouting.build_causal_window_self_attention_layout(lengths, sbs, case["window"])
        mask, mask_layout = bs.layouting.build_causal_window_self_attention_mask(lengths, layout, sbs, case["window"])
        return layout, dict(attention_mask=mask, sparsity_layout_mask=mask_layout)
    layout = _bigbird(heads, n, g)
    mask_layout = (layout & torch.ones((n, n), dtype=torch.bool, device=g.device).triu()).contiguous()
    where = mask_layout.nonzero()
    offsets = torch.arange(sbs, device=g.device)
    mask = ((where[:, 2] * sbs)[:, None, None] + offsets[None, None, :]
            > (where[:, 1] * sbs)[:, None, None] + offsets[None, :, None])
    return layout, dict(attention_mask=mask, sparsity_layout_mask=mask_layout)


def _blocks(count, sbs, dtype, g, scale=1.0):
    return (torch.randn((count, sbs, sbs), generator=g, device=g.device) * scale).to(DTYPES[dtype])


def prepare(case, seed):
    bs.utils.disable_validation()
    g = torch.Generator(device="cuda").manual_seed(seed)
    sbs, dtype, train = case["sbs"], case["dtype"], case.get("train", False)
    state = dict(case=case, cache={})
    if case["op"] == "attention":
        n, slices = case["seq"] // sbs, case["head_dim"] // sbs
        layout, extra = _attention_pattern(case, g)
        full = torch.ones((case["heads"], n, slices), dtype=torch.bool, device="cuda")
        count = case["heads"] * n * slices
        state.update(layout=layout, extra=extra, full=full, inputs=[_blocks(count, sbs, dtype, g) for _ in range(3)])
        if train:
            # query blocks that attend to nothing (padding) have no output block
            layout_o = bs.layouting.build_sparsity_layout_matmul(layout, full)
            state["grad"] = _blocks(int(layout_o.sum()), sbs, dtype, g)
    elif case["op"] == "matmul":
        rows, inner, cols = case["m"] // sbs, case["k"] // sbs, case["n"] // sbs
        order = _shuffled(inner, g)
        layout_x = _bernoulli((case["batch"], rows, inner), case["density"], 1)
        layout_x = layout_x[:, _shuffled(rows, g)][:, :, order].contiguous()
        layout_y = _bernoulli((case["batch"], inner, cols), case["density"], 2)
        layout_y = layout_y[:, order][:, :, _shuffled(cols, g)].contiguous()
        layout_o = bs.layouting.build_sparsity_layout_matmul(layout_x, layout_y)
        state.update(layout_x=layout_x, layout_y=layout_y, layout_o=layout_o,
                     inputs=[_blocks(int(layout_x.sum()), sbs, dtype, g, 1 / math.sqrt(case["k"])),
                             _blocks(int(layout_y.sum()), sbs, dtype, g)])
        if train:
            state["grad"] = _blocks(int(layout_o.sum()), sbs, dtype, g, 1 / math.sqrt(case["n"]))
    elif case["op"] == "softmax":
        n = case["n"] // sbs
        lower = torch.ones((n, n), dtype=torch.bool, device="cuda").tril()
        layout = lower | _bernoulli((case["batch"], n, n), case["density"], 1)
        layout = layout[_shuffled(case["batch"], g)].contiguous()
        count = int(layout.sum())
        state.update(layout=layout, inputs=[_blocks(count, sbs, dtype, g, 2.0)])
        if train:
            state["grad"] = _blocks(count, sbs, dtype, g)
    else:
        layout = _bernoulli((case["batch"], case["m"] // sbs, case["n"] // sbs), case["density"], 1)
        layout = layout[:, _shuffled(case["m"] // sbs, g)].contiguous()
        dense = torch.randn((case["batch"], case["m"], case["n"]), generator=g, device="cuda").to(DTYPES[dtype])
        blocks = dense.view(case["batch"], case["m"] // sbs, sbs, case["n"] // sbs, sbs)
        blocks.mul_(layout[:, :, None, :, None])
        state["inputs"] = [dense]
    if train:
        for tensor in state["inputs"]:
            tensor.requires_grad_(True)
    return state


# ---------------------------------------------------------------------------------------------------- one pass

def run(state):
    case = state["case"]
    sbs, inputs = case["sbs"], state["inputs"]
    if case["op"] == "attention":
        full = state["full"]
        q, k, v = inputs
        out = bs.ops.flash_attention(q, full, k, full, v, full, state["layout"], sbs, layout_cache=state["cache"],
                                     **state["extra"])
    elif case["op"] == "matmul":
        x, y = inputs
        out = bs.ops.matmul(x, state["layout_x"], y, state["layout_y"], state["layout_o"], sbs,
                            layout_cache=state["cache"])
    elif case["op"] == "softmax":
        out = bs.ops.softmax(inputs[0], state["layout"], sbs, layout_cache=state["cache"])
    else:
        layout = bs.layouting.build_sparsity_layout(inputs[0], sbs)
        compressed = bs.ops.to_sparse(inputs[0], layout, sbs)
        return layout, compressed, bs.ops.to_dense(compressed, layout, sbs)
    if not case["train"]:
        return out
    return (out.detach(), *torch.autograd.grad(out, inputs, state["grad"]))


# ---------------------------------------------------------------------------------------------------- the least work

@functools.lru_cache(maxsize=None)
def _expected_pairs(sbs, seq, heads, pattern, density, window):
    """Block pairs in which some score counts, and mask bytes, over all heads (expected over the random parts)."""
    n = seq // sbs
    if pattern == "bernoulli":
        return heads * n * n * density, 0
    if pattern == "bigbird":
        layout = _bigbird(1, n, torch.Generator().manual_seed(0))[0]
        return heads * int(layout.tril().sum()), heads * int(layout.tril().triu().sum()) * sbs * sbs
    # padded sequences use three quarters of the positions on average
    used = [max(round(n * share), 1) for share in (0.55, 0.65, 0.75, 0.85, 0.95)]
    reach = n if pattern == "causal" else -(-(window - 1) // sbs)
    pairs = sum(min(i, reach) + 1 for last in used for i in range(last)) / len(used)
    return heads * pairs, (0 if pattern == "causal" else heads * 2 * 0.75 * n * sbs * sbs)


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    sbs, train = case["sbs"], case.get("train", False)
    if case["op"] == "attention":
        pairs, mask_bytes = _expected_pairs(sbs, case["seq"], case["heads"], case["pattern"],
                                            case.get("density", 0), case.get("window", 0))
        tensor = case["heads"] * case["seq"] * case["head_dim"] * size
        # Q, K, V in, O out; a training step also dO in and three gradients out, and five more products
        return dict(bytes=(8 if train else 4) * tensor + mask_bytes,
                    flops=pairs * sbs * sbs * case["head_dim"] * (14 if train else 4))
    if case["op"] == "matmul":
        density = case["density"]
        rows, inner, cols = case["m"] // sbs, case["k"] // sbs, case["n"] // sbs
        pairs = case["batch"] * rows * inner * cols * density ** 2
        blocks = (rows * inner + inner * cols) * density + rows * cols * (1 - (1 - density ** 2) ** inner)
        return dict(bytes=(2 if train else 1) * case["batch"] * blocks * sbs * sbs * size,
                    flops=(3 if train else 1) * pairs * 2 * sbs ** 3)
    if case["op"] == "softmax":
        n = case["n"] // sbs
        blocks = case["batch"] * (n * (n + 1) / 2 + n * (n - 1) / 2 * case["density"])
        return dict(bytes=(4 if train else 2) * blocks * sbs * sbs * size, flops=(9 if train else 5) * blocks * sbs * sbs)
    dense = case["batch"] * case["m"] * case["n"] * size
    # the dense tensor is read to find the layout, its active blocks are written, and the dense result is written
    return dict(bytes=dense * (2 + case["density"]), flops=0)


def tolerance(case):
    """About four times the largest relative error seen against the same path in 64 bits on the dense tensors: attention
    5e-7 to 9e-7 in fp32, 3.1e-4 in fp16 and 2.5e-3 in bf16 (probabilities are rounded before they multiply the
    values), products 5.9e-7, 2.1e-4 and 1.7e-3, softmax 8.8e-8."""
    if case["op"] == "convert":
        return "exact"
    if case["op"] == "softmax":
        return {"rel": 4e-7}
    if case["op"] == "attention":
        return {"rel": {"fp32": 4e-6, "fp16": 1.2e-3, "bf16": 1e-2}[case["dtype"]]}
    return {"rel": {"fp32": 2.4e-6, "fp16": 8e-4, "bf16": 7e-3}[case["dtype"]]}

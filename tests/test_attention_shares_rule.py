"""Which attention layouts get shares (attn_shares_piece): those that were measured to gain, and none that were not."""

import ctypes

import pytest
import torch

from blksprs_amd import _capi


def _layout(kind, heads, blocks):
    if kind == "causal":
        return torch.ones((blocks, blocks), dtype=torch.bool).tril().expand(heads, blocks, blocks)
    i = torch.arange(blocks)
    fixed = ((i[:, None] - i[None, :]).abs() <= 4) | (i[:, None] < 2) | (i[None, :] < 2)
    chosen = torch.rand((heads, blocks, blocks), generator=torch.Generator().manual_seed(1)).argsort(dim=-1)[..., :3]
    return torch.zeros((heads, blocks, blocks), dtype=torch.bool).scatter_(2, chosen, True) | fixed


# GPU time of forward and backward without -> with shares, us
@pytest.mark.parametrize("dtype,sbs,head_dim,heads,seq,kind,wanted", [
    (torch.float32, 32, 64, 8, 2048, "causal", False),  # 180 -> 197
    (torch.float32, 64, 64, 8, 2048, "causal", False),  # 178 -> 193
    (torch.float32, 32, 64, 4, 2048, "causal", True),  # 162 -> 146
    (torch.float32, 32, 64, 2, 4096, "causal", True),  # 292 -> 206
    (torch.float32, 32, 128, 4, 2048, "causal", True),  # 307 -> 291
    (torch.float32, 64, 64, 1, 6080, "causal", True),  # 425 -> 274 (a call)
    (torch.float32, 16, 64, 4, 2048, "causal", False),  # 142 -> 146
    (torch.float32, 16, 64, 2, 4096, "causal", True),  # 260 -> 242
    (torch.bfloat16, 32, 64, 8, 2048, "causal", False),  # 57 -> 57
    (torch.bfloat16, 32, 64, 2, 4096, "causal", False),  # 76 -> 84
    (torch.bfloat16, 32, 64, 24, 1536, "causal", True),  # 80 -> 63
    (torch.bfloat16, 32, 128, 24, 1536, "causal", False),  # 134 -> 137
    (torch.float16, 16, 64, 8, 2048, "causal", True),  # 95 -> 70
    (torch.float16, 16, 64, 4, 2048, "causal", False),  # 56 -> 57
    (torch.float16, 16, 64, 24, 1536, "causal", False),  # 85 -> 87
    (torch.float32, 32, 64, 8, 2048, "bigbird", True),  # 196 -> 137
    (torch.float32, 32, 64, 16, 1024, "bigbird", False),  # 121 -> 125
    (torch.float32, 32, 64, 24, 1536, "bigbird", True),  # 275 -> 215
    (torch.float32, 32, 128, 24, 1536, "bigbird", False),  # 630 -> 642
    (torch.float32, 32, 128, 14, 1056, "bigbird", True),  # 334 -> 239 (a call)
    (torch.float32, 64, 128, 6, 1664, "bigbird", True),  # 382 -> 330
    (torch.float32, 32, 64, 12, 2048, "causal", False),  # 221 -> 243
    (torch.float32, 32, 64, 2, 4096, "bigbird", True),  # 331 -> 104
    (torch.bfloat16, 32, 64, 8, 2048, "bigbird", False),  # 65 -> 64
    (torch.bfloat16, 32, 64, 24, 1536, "bigbird", True),  # 104 -> 76
    (torch.bfloat16, 32, 64, 2, 4096, "bigbird", True),  # 107 -> 49
    (torch.bfloat16, 32, 96, 7, 3328, "bigbird", True),  # 75 -> 29 (forward)
    (torch.float16, 16, 64, 4, 2048, "bigbird", False),  # 74 -> 72
])
def test_layouts_that_get_shares(dtype, sbs, head_dim, heads, seq, kind, wanted):
    assert _wanted(dtype, sbs, head_dim, heads, seq, kind, 0) == wanted


# a call without a cache, without -> with shares, us
@pytest.mark.parametrize("dtype,sbs,head_dim,heads,seq,kind,wanted", [
    (torch.float32, 64, 64, 1, 6080, "causal", True),  # 600 -> 554
    (torch.float32, 32, 64, 8, 2048, "bigbird", False),
    (torch.float32, 32, 128, 14, 1056, "bigbird", False),  # 479 -> 484
    (torch.float16, 16, 64, 5, 3152, "causal", False),  # 373 -> 460
    (torch.bfloat16, 32, 96, 7, 3328, "bigbird", False),  # 237 -> 265
])
def test_layouts_that_get_shares_for_one_call(dtype, sbs, head_dim, heads, seq, kind, wanted):
    assert _wanted(dtype, sbs, head_dim, heads, seq, kind, _capi.SHARES_FOR_ONE_CALL) == wanted


def _wanted(dtype, sbs, head_dim, heads, seq, kind, flag):
    blocks = seq // sbs
    layout = _layout(kind, heads, blocks)
    a = _capi.AttnArgs()
    a.B, a.nq, a.nk, a.nh, a.nhv = heads, blocks, blocks, head_dim // sbs, head_dim // sbs
    a.sbs, a.dtype = sbs, _capi.DTYPE_CODES[dtype]
    piece, most_groups, most_merges = _capi.c_int64(), _capi.c_int64(), _capi.c_int64()
    rc = _capi.load().bsa_attn_shares_piece(ctypes.byref(a), flag, int(layout.sum()), int(layout.sum(2).max()), ctypes.byref(piece),
                                            ctypes.byref(most_groups), ctypes.byref(most_merges))
    assert rc == 0
    return piece.value > 0

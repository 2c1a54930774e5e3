"""The attention kernels for blocks of 16 and 32 (attn_small_fwd.hip, attn_small_bwd.hip) at the edges of their
tiles and of their dispatch: every number of head slices they are built for and one more, different numbers for q / k
and v, key lists of one block, of a step and one more, of more than the 64 entries of a window, launches small and
large enough for every way of sharing a list between waves."""

import pytest
import torch

import blksprs_amd as bs
from oracle import blksprs_oracle as orc
from tests.test_attention_gpu import TOL, _run_case, assert_close, rand_blocks

pytestmark = pytest.mark.gpu


DTYPES = [torch.float16, torch.bfloat16, torch.float32]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sbs,nh,nhv", [(16, n, n) for n in range(1, 10)] + [(32, n, n) for n in range(1, 6)]
                         + [(16, 3, 5), (16, 6, 2), (32, 1, 3), (32, 4, 2)])
def test_head_slices(device, dtype, sbs, nh, nhv):
    _run_case(device, dtype, sbs, B=2, nq=3, nk=5, nh=nh, nhv=nhv, density=0.6, seed=10 * nh + nhv)
    _run_case(device, dtype, sbs, B=1, nq=3, nk=5, nh=nh, nhv=nhv, density=0.6, seed=nh + nhv, use_mask=True,
              use_bias=True, sparse_heads=True, custom_o=True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sbs", [16, 32])
@pytest.mark.parametrize("nk", [1, 4, 5, 63, 64, 65, 150])
def test_list_lengths(device, dtype, sbs, nk):
    _run_case(device, dtype, sbs, B=1, nq=2, nk=nk, nh=2, nhv=2, density=1.0, seed=nk)
    _run_case(device, dtype, sbs, B=1, nq=5, nk=nk, nh=2, nhv=2, density=0.5, seed=nk + 1, use_mask=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sbs", [16, 32])
@pytest.mark.parametrize("B,n", [(1, 70), (9, 64), (140, 60)])
@pytest.mark.parametrize("use_causal", [False, True])
def test_rows_of_a_launch(device, dtype, sbs, B, n, use_causal):
    """70, 576 and 8400 query blocks: four, two and one wave per query block (and per key block)."""
    nk = n if use_causal else 3
    _run_case(device, dtype, sbs, B=B, nq=n, nk=nk, nh=1, nhv=1, density=0.1 if use_causal else 0.6,
              seed=B + n, use_causal=use_causal)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nh", [1, 2, 3, 4])
@pytest.mark.parametrize("B,n", [(1, 3), (2, 9), (33, 16)])
def test_sums_of_waves_that_share_a_key_block(device, dtype, nh, B, n):
    """dK and dV of 16-bit blocks of 32 are larger than the tiles of the wave that has them: lists of one step and of several
    for each of four waves (3 and 18 key blocks) and of two (528)."""
    _run_case(device, dtype, 32, B=B, nq=n, nk=n, nh=nh, nhv=nh, density=0.8, seed=10 * nh + n, use_mask=True)
    _run_case(device, dtype, 32, B=B, nq=n, nk=n, nh=nh, nhv=nh, density=0.3, seed=nh + n, use_causal=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,n", [(2, 1), (7, 7), (8, 8), (8, 9), (13, 17), (16, 3), (20, 11)])
def test_rows_over_xcds(device, dtype, B, n):
    """Whole batch entries of an XCD, entries shared by all eight, last rows that are no multiple of eight."""
    _run_case(device, dtype, 16, B=B, nq=n, nk=n, nh=2, nhv=2, density=0.5, seed=100 * B + n)
    _run_case(device, dtype, 16, B=B, nq=n, nk=n, nh=1, nhv=1, density=0.5, seed=100 * B + n, use_causal=True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sbs", [16, 32])
def test_tensors_that_start_inside_a_16_byte_piece(device, dtype, sbs):
    """Operands, output gradient and mask as contiguous views one element into a larger buffer: the kernels that move
    16 bytes at a time leave them to the ones that load through registers, forward and backward, one by one."""
    def inside(t):
        buffer = torch.empty(t.numel() + 1, dtype=t.dtype, device=device)
        view = buffer[1:].view(t.shape).copy_(t)
        assert view.is_contiguous() and view.data_ptr() % 16 == t.element_size()
        return view

    g = torch.Generator().manual_seed(sbs)
    B, n, nh = 2, 5, 2
    la = orc.random_layout((B, n, n), 0.6, g, ensure_rows=True)
    full = torch.ones((B, n, nh), dtype=torch.bool)
    q, k, v, go = (rand_blocks(B * n * nh, sbs, dtype, sbs + i) for i in range(4))
    mask = torch.rand((int(la.sum()), sbs, sbs), generator=g) < 0.3
    r64 = [t.double().requires_grad_(True) for t in (q, k, v)]
    ref = orc.flash_attention(r64[0], full.numpy(), r64[1], full.numpy(), r64[2], full.numpy(), la.numpy(), sbs, mask=mask,
                              layout_mask=la.numpy(), acc_dtype=torch.float64)
    ref.backward(go.double())
    fd, ld = full.to(device), la.to(device)
    for which in ("q", "k", "v", "go", "mask", "all"):
        place = lambda name, t: inside(t) if which in (name, "all") else t.to(device)
        ops = [place(name, t).detach().requires_grad_(True) for name, t in zip("qkv", (q, k, v))]
        out = bs.ops.flash_attention(ops[0], fd, ops[1], fd, ops[2], fd, ld, sbs, attention_mask=place("mask", mask),
                                     sparsity_layout_mask=ld)
        out.backward(place("go", go))
        for name, got, want in zip(("O", "dQ", "dK", "dV"), (out, *(t.grad for t in ops)), (ref, *(t.grad for t in r64))):
            assert_close(got, want, TOL[dtype], f"{name}, {which} inside a piece")

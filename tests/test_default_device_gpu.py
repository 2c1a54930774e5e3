"""Programs whose default device is the GPU: what the host itself reads stays in its own memory."""

import threading

import pytest
import torch

import blksprs_amd as bs

pytestmark = pytest.mark.gpu


def _convert(device):
    layout = torch.zeros((2, 4, 4), dtype=torch.bool)
    layout[:, 1:, ::2] = True
    x = torch.arange(2 * 64 * 64, dtype=torch.float32).view(2, 64, 64)
    blocks = x.view(2, 4, 16, 4, 16).permute(0, 1, 3, 2, 4)[layout]
    assert torch.equal(torch.Tensor(bs.ops.to_sparse(x, layout, 16)), blocks)


def _attend(device):
    full = torch.ones((2, 3, 1), dtype=torch.bool)
    layout = torch.ones((3, 3), dtype=torch.bool).tril().expand(2, 3, 3).contiguous()
    q, k, v = (torch.randn(6, 16, 16) for _ in range(3))
    lengths = torch.tensor([48, 20])
    out = torch.Tensor(bs.ops.flash_attention(q, full, k, full, v, full, layout, 16, causal_lengths=lengths)).view(2, 48, 16)
    scores = torch.matmul(q.double().view(2, 48, 16).cpu(), k.double().view(2, 48, 16).cpu().transpose(1, 2).contiguous()) / 4
    positions = torch.arange(48, device="cpu")
    seen = (positions[None, :] <= positions[:, None])[None] & (positions[None, None, :] < lengths.cpu()[:, None, None])
    want = scores.masked_fill(~seen, float("-inf")).softmax(-1) @ v.double().view(2, 48, 16).cpu()
    for b, length in enumerate((48, 20)):
        error = out[b, :length].double().cpu() - want[b, :length]
        assert float(error.norm()) <= 4e-6 * float(want[b, :length].norm())  # 32-bit sums leave 5e-7 to 9e-7


@pytest.mark.parametrize("call", [_convert, _attend])
def test_calls_under_a_default_device(device, call):
    failures = []

    def program():  # a thread of its own: what a thread has pinned before, it uses again
        try:
            with torch.device(device):
                call(device)
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    thread = threading.Thread(target=program)
    thread.start()
    thread.join()
    if failures:
        raise failures[0]

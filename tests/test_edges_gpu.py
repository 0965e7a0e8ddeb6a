"""Edges of the kernels' tile and dispatch ranges against the oracle or an fp64 reference: remainders,
smallest and largest sizes of a rule, and operands that take the general path next to ones that do not."""

import pytest
import torch

from oracle import llama_q4_ref as R
from q4llm import ops

pytestmark = pytest.mark.gpu


def misaligned(t):
    """A contiguous copy of t whose data starts 4 bytes past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 4, dtype=t.dtype, device=t.device)
    out = buf[1:1 + t.numel()].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == 4 and out.is_contiguous()
    return out


@pytest.mark.parametrize("n,k,group", [(1, 8, 8), (3, 48, 16), (5, 32, 32), (7, 320, 64), (33, 384, 128), (130, 256, 256),
                                       (9, 1536, 512), (2, 1024, 1024), (5, 288, 96)])
def test_quantize_word_and_group_paths(dev, n, k, group):
    """One thread per word (power-of-two groups up to 512, 16-byte aligned w) and one per group (the
    rest) give the oracle's bits; zero groups, exact ties and the clamp's ends among the inputs."""
    g = torch.Generator().manual_seed(n + k + group)
    w = torch.randn(n, k, generator=g)
    w[0, :8] = torch.tensor([7.0, -7.0, 0.5, 1.5, -0.5, -1.5, 2.5, -8.5])
    w[-1, -8:] = 0.0
    qw, sc = R.quantize_q4(w, group)
    for wd in (w.to(dev), misaligned(w.to(dev))):
        got_q, got_s = ops.quantize_q4(wd, group)
        assert torch.equal(got_q.cpu(), qw) and torch.equal(got_s.cpu().view(torch.int16), sc.view(torch.int16))


@pytest.mark.parametrize("group", [8, 64, 512])
def test_quantize_non_finite_same_on_both_paths(dev, group):
    w = torch.randn(8, 512, device=dev)
    w[0, 3], w[1, 70], w[2, 500], w[3, :] = float("inf"), float("nan"), float("-inf"), float("nan")
    a, b = ops.quantize_q4(w, group), ops.quantize_q4(misaligned(w), group)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1].view(torch.int16), b[1].view(torch.int16))

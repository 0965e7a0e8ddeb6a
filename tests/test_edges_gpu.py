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


def linear_case(dev, M, N, K, group, seed):
    g = torch.Generator().manual_seed(seed)
    qw, sc = R.quantize_q4(torch.randn(N, K, generator=g) * 0.02, group)
    x, res = torch.randn(M, K, generator=g), torch.randn(M, N, generator=g)
    w = R.dequantize_q4(qw, sc, group).double()
    ref = x.double() @ w.t() + res.double()
    # x = hi + lo up to 2^-22 |x|; fp32 sums of at most two adds per 32 k, a scale per group and the
    # waves' and residual's adds, each rounding by 2^-24 of a partial sum that sum |x w| + |res| bounds
    bound = ((x.double().abs() @ w.abs().t()) + res.double().abs()) * (2.0 ** -22 + (K / 16 + K / group + 32) * 2.0 ** -24)
    return x.to(dev), qw.to(dev), sc.to(dev), res.to(dev), ref, bound


@pytest.mark.parametrize("M,N,K,group", [(2, 1, 64, 32), (16, 15, 192, 64), (17, 33, 96 * 4, 96), (9, 4097, 256, 128),
                                         (32, 4112, 128, 32), (3, 8193, 192, 32), (31, 8208, 384, 384), (1, 16, 4160, 64),
                                         (32, 48, 4096, 128), (16, 17, 8192, 256), (33, 48, 4096, 128), (17, 16, 4160, 32)])
def test_linear_few_rows(dev, M, N, K, group):
    """The one-launch kernel for few rows at the edges of its column counts (16, 32 and 64 per workgroup),
    K remainders (64 of a 128-k step, fewer steps than waves), groups (any multiple of 32) and its
    largest M, and the sizes just past its rule; the residual aliasing y, with and without a workspace."""
    x, qw, sc, res, ref, bound = linear_case(dev, M, N, K, group, M * 1000 + N)
    for fn in (ops.q4_linear, ops.q4_linear_ws):
        y = torch.full((M, N), float("nan"), device=dev)
        fn(x, qw, sc, group, out=y)
        assert ((y.cpu().double() - (ref - res.cpu().double())).abs() <= bound).all(), (fn, M, N, K, group)
        h = res.clone()
        fn(x, qw, sc, group, residual=h, out=h)
        assert ((h.cpu().double() - ref).abs() <= bound).all(), (fn, M, N, K, group)


@pytest.mark.parametrize("M,N,K,group", [(33, 40, 128, 32), (100, 515, 3072, 32), (257, 256, 256, 128), (300, 1030, 2048, 64),
                                         (385, 260, 4096, 256), (513, 3072, 1024, 128), (640, 5120, 192, 64),
                                         (1024, 4100, 512, 128)])
def test_linear_many_rows(dev, M, N, K, group):
    """q4_linear through its workspace: both pipelined tiles with ragged rows and columns, K splits past
    256 rows, an exact-planes workspace (no split), and a residual aliasing y."""
    x, qw, sc, res, ref, bound = linear_case(dev, M, N, K, group, M + N)
    y = torch.full((M, N), float("nan"), device=dev)
    ops.q4_linear(x, qw, sc, group, out=y)
    assert ((y.cpu().double() - (ref - res.cpu().double())).abs() <= bound).all()
    for split in (False, True):
        h = res.clone()
        need = ops.q4_linear_ws_split_bytes(M, N, K, group) if split else 4 * M * K
        ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=dev)
        ops.q4_linear_ws(x, qw, sc, group, residual=h, out=h, workspace=ws)
        assert ((h.cpu().double() - ref).abs() <= bound).all(), split

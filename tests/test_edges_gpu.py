"""Edges of the kernels' tile and dispatch ranges against the oracle or an fp64 reference: remainders,
smallest and largest sizes of a rule, and operands that take the general path next to ones that do not."""

import pytest
import torch

from oracle import llama_q4_ref as R
from q4llm import ops
from q4llm._lib import LIB

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


@pytest.mark.parametrize("M,N,K,group", [(16, 520, 14336, 128), (2, 264, 28672, 64), (32, 64, 4096, 128), (12, 33000, 256, 32),
                                         (20, 33000, 192, 64), (5, 8448, 16384, 128)])
def test_linear_few_rows_on_tiles(dev, M, N, K, group):
    """Few rows past the line of the one-launch kernel (long K, many columns), which run on the tiles when the
    workspace holds their partials: every row and column of a tile that is mostly padding."""
    x, qw, sc, res, ref, bound = linear_case(dev, M, N, K, group, M + N)
    y = ops.q4_linear_ws(x, qw, sc, group, split=True)
    assert ((y.cpu().double() - (ref - res.cpu().double())).abs() <= bound).all()
    h = res.clone()
    ops.q4_linear_ws(x, qw, sc, group, residual=h, out=h, split=True)
    assert ((h.cpu().double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("M,N,K,group", [(33, 40, 128, 32), (100, 515, 3072, 32), (257, 256, 256, 128), (300, 1030, 2048, 64),
                                         (385, 260, 4096, 256), (513, 3072, 1024, 128), (640, 5120, 192, 64),
                                         (1024, 4100, 512, 128), (19, 819, 6144, 128), (35, 1225, 3904, 64), (250, 3560, 128, 128),
                                         (700, 3560, 128, 32), (250, 3560, 384, 128), (33, 257, 64, 64), (257, 401, 4160, 32), (1013, 1270, 192, 32),
                                         (512, 2047, 256, 128), (512, 1025, 256, 64)])
def test_linear_many_rows(dev, M, N, K, group):
    """q4_linear through its workspace: both pipelined tiles with ragged rows and columns, K splits (also of
    M N that is no multiple of four), the shortest K on both sides of the line to the one-launch kernel, an
    exact-planes workspace (no split), and a residual aliasing y."""
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


@pytest.mark.parametrize("M,N,K,group", [(33, 200, 384, 128), (100, 257, 320, 64), (300, 515, 1152, 128), (9, 40, 384, 128),
                                         (40, 96, 96 * 2, 32 * 3)])
def test_linear_scales_off_a_word(dev, M, N, K, group):
    """Rows 1.. of a weight with an odd number of groups: its scales start between two words, which the
    kernel that loads them by words must not take."""
    x, qw, sc, res, ref, bound = linear_case(dev, M, N + 1, K, group, M + N)
    ref, bound, qw, sc, res = ref[:, 1:], bound[:, 1:], qw[1:], sc[1:], res[:, 1:].contiguous()
    if K // group % 2:
        assert sc.data_ptr() % 4 == 2
    for fn in (ops.q4_linear, ops.q4_linear_ws):
        y = fn(x, qw, sc, group, residual=res)
        assert ((y.cpu().double() - ref).abs() <= bound).all(), fn
        y = torch.full((M, N), float("nan"), device=dev)
        fn(x, qw, sc, group, out=y)
        assert ((y.cpu().double() - (ref - res.cpu().double())).abs() <= bound).all(), fn


def attn_ref64(q, kc, vc, start, scale):
    C, nq, hd = q.shape
    n, nkv = min(start + C, kc.shape[0]), kc.shape[1]
    g = nq // nkv
    mask = torch.arange(n)[None, :] > (start + torch.arange(C))[:, None]
    out = torch.empty(C, nq, hd, dtype=torch.float64)
    for h in range(nq):
        s = (q[:, h].double() @ kc[:n, h // g].double().t()) * scale
        out[:, h] = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ vc[:n, h // g].double()
    return out.reshape(C, nq * hd)


@pytest.mark.parametrize("C,start,L,nq,nkv,hd,ps", [
    (2, 0, 33, 8, 8, 64, None), (33, 31, 96, 6, 2, 128, None), (31, 480, 512, 5, 1, 64, None),
    (65, 0, 65, 24, 8, 128, None), (256, 1792, 2048, 24, 8, 128, None), (97, 3900, 4096, 7, 1, 128, None),
    (64, 700, 777, 8, 1, 64, None), (256, 0, 256, 4, 2, 64, 32), (130, 125, 256, 12, 12, 64, 96),
    (96, 416, 512, 24, 8, 128, 512), (40, 20, 300, 20, 4, 128, 32)])
@pytest.mark.parametrize("scale", [0.088, -0.3, 0.0, 4.0])
def test_attn_prefill_units_and_splits(dev, kernel_override, C, start, L, nq, nkv, hd, ps, scale):
    """Chunks whose 32-row units do not divide over the workgroups' waves, rows and keys off the 32-key
    blocks, one and many splits, splits that some rows of a workgroup do not reach, and scales of both
    signs, zero, and one whose maxima grow by more than the rescaling threshold."""
    if ps:
        kernel_override("attn_ps", ps)
    g = torch.Generator().manual_seed(C + start + L)
    q = torch.randn(C, nq, hd, generator=g)
    kc, vc = torch.randn(L, nkv, hd, generator=g).half(), torch.randn(L, nkv, hd, generator=g).half()
    kc[: min(64, L)] *= 0.05  # small scores first: the running maximum grows in later blocks
    kc[start + C:], vc[start + C:] = 100.0, 1000.0  # stale rows past every position: no weight
    ref = attn_ref64(q, kc, vc, start, scale)
    out = torch.full((C, nq * hd), float("nan"), device=dev)
    ops.attn_bucket(q.to(dev), kc.to(dev), vc.to(dev), L, torch.tensor([start], dtype=torch.int32, device=dev), scale,
                    out=out)
    # scores of fp16 hi + lo queries: 2^-22 sum |q k| each, the same again for the fp32 sums; P likewise
    smax = (q.abs().double().sum(-1).max() * 4.0 * abs(scale)).item()
    assert (out.cpu().double() - ref).abs().max().item() <= 5.0 * (2.0 ** -20 * max(smax, 1.0)) + 1e-6


@pytest.mark.parametrize("M,N,K", [(511, 3076, 2056), (512, 3076, 2056), (257, 2052, 8192), (700, 2243, 3000),
                                   (2049, 1030, 1032), (33, 8196, 8200), (1023, 513, 4104), (2600, 3000, 264),
                                   (2, 4096, 65536), (1536, 1540, 4096), (4096, 2052, 64)])
def test_gemm_plan_and_workspace_sizes(dev, M, N, K):
    """Sizes on both sides of the GEMM rule's lines (latency-bound, the tiles chosen by estimated time, the K
    split), each with the workspace it asks for, with one that only a smaller plan fits, and with none where
    the split by size alone needs none."""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randn(M, K, device=dev, generator=g).half()
    b = torch.randn(N, K, device=dev, generator=g).half()
    ref = a.double() @ b.double().t()
    # fp32 sums of K products (their errors add like a random walk; 8 sigma) and the fp16 result
    bound = 2.0 ** -11 * ref.abs() + 8 * K ** 0.5 * 2.0 ** -24 * (K ** 0.5) + 2.0 ** -14
    f = LIB.raw("gemm_f16_nt_ws")
    st = torch.cuda.current_stream(dev).cuda_stream

    def check(c, what):
        assert ((c.double() - ref).abs() <= bound).all(), what

    check(ops.gemm_f16_nt(a, b), "no workspace entry")
    need = ops.gemm_f16_nt_ws_bytes(M, N, K)
    for nbytes in {need, max(need, 16) + 48, need // 2, 0} if M >= 512 else {need, need + 48}:
        ws = torch.full((nbytes + 64,), 255, dtype=torch.uint8, device=dev)
        c = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
        assert f(ops.ptr(a), ops.ptr(b), ops.ptr(c), M, N, K, K, K, N, ops.ptr(ws) if nbytes else None, nbytes, st) == 0
        check(c, nbytes)
        assert (ws[nbytes:] == 255).all()
    check(ops.gemm_f16_nt_ws(a, b), "its own workspace")


@pytest.mark.parametrize("M,N,K", [(512, 1024, 1024), (4096, 64, 4096), (1000, 256, 2048), (511, 1024, 4096), (256, 3072, 8192),
                                   (512, 3072, 8192), (513, 1024, 4096)])
def test_gemm_workspace_contract(dev, monkeypatch, M, N, K):
    """Which workspaces gemm_f16_nt_ws takes, on both sides of 512 rows and 4 GFLOP: the size it asks for and
    more always; less, or none, only from both lines on. Without memory for a workspace the wrapper runs
    the form that needs none."""
    a, b = torch.ones(M, K, device=dev).half(), torch.ones(N, K, device=dev).half() / 64
    need = ops.gemm_f16_nt_ws_bytes(M, N, K)
    f = LIB.raw("gemm_f16_nt_ws")
    st = torch.cuda.current_stream(dev).cuda_stream
    lenient = M >= 512 and 2 * M * N * K >= 4e9
    assert need > 0
    for nbytes in (0, need // 2, need - 16, need, need + 64):
        ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=dev)
        c = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
        rc = f(ops.ptr(a), ops.ptr(b), ops.ptr(c), M, N, K, K, K, N, ops.ptr(ws) if nbytes else None, nbytes, st)
        assert rc == (0 if nbytes >= need or lenient else -5), nbytes
        assert rc != 0 or (c == K / 64).all()
    empty = torch.empty

    def no_workspace(*args, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no memory")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", no_workspace)
    assert (ops.gemm_f16_nt_ws(a, b) == K / 64).all()


def test_native_calls_match_python_wrappers(dev, monkeypatch):
    """The native calls and the Python wrappers they stand in for give the same bits and the same errors,
    on the current stream; operands the native code leaves alone (views that need a copy, an `out`, other
    shapes) still work."""
    from q4llm import llama_q4 as Q
    g = torch.Generator(device=dev).manual_seed(3)

    def rnd(*s):
        return torch.randn(*s, device=dev, generator=g)

    lin = Q.QLinear(rnd(96, 256) * 0.02, 32)
    qw, sc = lin.qweight, lin.scales
    x1, x5, x40, res = rnd(1, 256), rnd(5, 256), rnd(40, 256), rnd(40, 96)
    kc, vc, q = rnd(64, 2, 64).half(), rnd(64, 2, 64).half(), rnd(3, 4, 64)
    st = torch.tensor([5], dtype=torch.int32, device=dev)
    a, b = rnd(33, 64).half(), rnd(24, 128).half()[:, :64]
    ws = torch.empty(1 << 20, dtype=torch.uint8, device=dev)

    def results():
        side = torch.cuda.Stream(dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        out16 = torch.empty(96, dtype=torch.float16, device=dev)
        with torch.cuda.stream(side):
            r = [ops.q4_gemv(qw, sc, x1, 32), ops.q4_gemv(qw, sc, x1[0].half(), 32, out_dtype=torch.float16),
                 ops.q4_gemv(qw, sc, x1[0], 32, residual=res[0]), ops.q4_gemv(qw, sc, x1[0].half(), 32, out=out16),
                 ops.q4_gemv(qw, sc, rnd(256, 2)[:, 0] * 0 + x1[0], 32), lin(x1), lin(x1[0]), lin(x5, residual=res[:5]),
                 lin(x40, residual=res), lin(x40.half()), lin(x40[None]), lin(rnd(256, 40).t() * 0 + x40),
                 ops.q4_linear(x1, qw, sc, 32), ops.attn_bucket(q, kc, vc, 64, st, 0.1),
                 ops.attn_bucket(q[:1], kc, vc, 33, st, 0.1, workspace=ws),
                 ops.attn_bucket(q.transpose(0, 1).contiguous().transpose(0, 1), kc, vc, 64, st, 1),
                 ops.gemm_f16_nt(a, b), ops.gemm_f16_nt_ws(a, b, workspace=ws), ops.gemm_f16_nt(a[:1], b)]
        assert r[3] is out16
        torch.cuda.current_stream(dev).wait_stream(side)
        return r

    native = results()
    for name in ("_gemv", "linear_call", "_attn", "_gemm"):
        monkeypatch.setattr(ops, name, ops._left_to_python)
    for i, (u, v) in enumerate(zip(native, results())):
        assert u.shape == v.shape and u.dtype == v.dtype and torch.equal(u, v), i
    monkeypatch.undo()
    for bad in (lambda: ops.q4_gemv(qw, sc, x1.double(), 32), lambda: ops.q4_gemv(qw, sc, x1[:, :64], 32),
                lambda: ops.q4_gemv(qw, sc.float(), x1, 32), lambda: ops.q4_linear(x5[:, :128], qw, sc, 32),
                lambda: ops.gemm_f16_nt(a, b.float()), lambda: ops.gemm_f16_nt(a.t(), b),
                lambda: lin(x5, residual=res), lambda: ops.q4_gemv(qw, sc, x1, 48)):
        with pytest.raises(ValueError):
            bad()

"""Whole-model parity on the GPU: LlamaQ4.step and the runner against the CPU oracle on the tiny
configs (exact greedy tokens; logits within the reference's per-op tolerance
1e-3 * max(1, max|ref|), scripts/debug/op_test.py:74-77), plus graph replay consistency.
Both sides keep fp16 KV caches, so the logit difference comes from rare one-ulp rounding flips of
cache entries whose fp32 values differ in the last bits."""

import json
import pathlib

import pytest
import torch

from oracle import llama_q4_ref as R
from q4llm import llm_runner, synth
from q4llm.llama_q4 import LlamaQ4

pytestmark = pytest.mark.gpu
GOLD = pathlib.Path(__file__).parent / "golden"


def build_pair(cfg, group, max_ctx, seed=0, std=None):
    """Weights of std 0.2; past hidden size 1024 such that a projection's gain, std sqrt(hidden), stays that of
    1024 (6.4). Scores are q . k / sqrt(hd) of entries of that size: std gain^2 = 41, where one fp16 ulp
    (2^-11) of the differently rounded K entries moves a score by up to gain^2 2^-11 = 0.02 and the logits by
    less than their tolerance; at 0.2 and hidden 3072 (gain 11) the same flips move scores by 0.06."""
    std = std or min(0.2, 6.4 / cfg["hidden_size"] ** 0.5)
    sd = synth.SyntheticWeights(cfg, seed, std=std)
    dense = {k: sd[k] for k in sd.keys()}
    ours = LlamaQ4(None, group=group, max_ctx=max_ctx, sd=dense, cfg=cfg)
    ref = R.LlamaQ4Ref(cfg, dense, group=group, max_ctx=max_ctx, rope=(ours.cos.cpu(), ours.sin.cpu()))
    return ours, ref


# K-split projections (their ranges at 128 and 256 rows: test_prefill_deferred_partials_...)
SPLIT_DIMS = dict(hidden_size=2048, intermediate_size=4096, num_attention_heads=16, num_key_value_heads=8, head_dim=128)


def ranges(model, chunk, L):
    """K ranges of the qkv, o, gate/up and down projections of a chunk (0: gate/up with the SwiGLU epilogue)."""
    return [r for _, r in model.step_plan(chunk, L)]


def tol(ref):
    return 1e-3 * max(1.0, ref.abs().max().item())


def test_quantized_weights_bit_exact(dev):
    ours, ref = build_pair(synth.TINY, 32, 128)
    assert torch.equal(ours.embed.qweight.cpu(), ref.embed.qweight)
    for lo, lr in zip(ours.layers, ref.layers):
        for name in ("wqkv", "wo", "wgu", "wdown"):
            assert torch.equal(getattr(lo, name).qweight.cpu(), lr[name].qweight), name
            assert torch.equal(getattr(lo, name).scales.cpu().view(torch.int16), lr[name].scales.view(torch.int16))


def test_step_prefill_and_decode_vs_oracle(dev):
    ours, ref = build_pair(synth.TINY, 32, 128)
    prompt = synth.prompt_ids(16, 1024, seed=0)
    ours_c, ref_c = ours.new_caches(), ref.new_caches()
    toks = torch.tensor([prompt], dtype=torch.int32)
    n1, l1 = ours.step(toks, torch.tensor([0], dtype=torch.int32), torch.tensor([15], dtype=torch.int32), ours_c, 64)
    r1, rl1 = ref.step(toks, torch.tensor([0], dtype=torch.int32), torch.tensor([15], dtype=torch.int32), ref_c, 64)
    assert int(n1.item()) == int(r1.item())
    assert (l1.cpu() - rl1).abs().max().item() <= tol(rl1)
    # Caches written in place: both sides round fp32 K/V to fp16; fp32 differences in the last bits
    # (growing slightly through the layers) flip a few roundings. Layer 0 differs by at most one
    # fp16 ulp where the value is not tiny; every layer stays within 2e-3 of the cache's max.
    for i in range(8):
        a, b = ours_c[i].cpu(), ref_c[i]
        if i < 2:
            big = b.float().abs() >= 2.0 ** -6
            ulps = (a.view(torch.int16).int() - b.view(torch.int16).int()).abs()
            assert ulps[big].max().item() <= 1
        assert (a.float() - b.float()).abs().max().item() <= 2e-3 * b.float().abs().max().item()
    nxt, rn = n1, r1
    for pos in range(16, 24):
        nxt, lg = ours.step(nxt.reshape(1, 1).cpu(), torch.tensor([pos], dtype=torch.int32),
                            torch.tensor([0], dtype=torch.int32), ours_c, 64)
        rn, rlg = ref.step(rn.reshape(1, 1), torch.tensor([pos], dtype=torch.int32), torch.tensor([0], dtype=torch.int32),
                           ref_c, 64)
        assert int(nxt.item()) == int(rn.item())
        assert (lg.cpu() - rlg).abs().max().item() <= tol(rlg)


@pytest.mark.parametrize("variant", ["baseline_std0.02", "std0.2"])
def test_tiny_generation_matches_golden(dev, variant):
    """16-token prompt, 32 greedy tokens, buckets {64, 128}, chunk 16 (weights
    N(0, 0.02) as stated, and N(0, 0.2) whose greedy tokens vary)."""
    gold = json.loads((GOLD / "tiny_tokens.json").read_text())[variant]
    sd = synth.SyntheticWeights(synth.TINY, gold["seed"], std=gold["std"])
    model = LlamaQ4(None, group=gold["group"], max_ctx=gold["max_ctx"], sd=sd, cfg=synth.TINY)
    res = llm_runner.run(model, gold["prompt"], gold["max_new_tokens"], gold["chunk"], gold["buckets"])
    assert res["tokens"] == gold["tokens"]
    assert res["new_tokens"] == gold["max_new_tokens"] and res["decode_steps"] == gold["max_new_tokens"] - 1


def test_generation_fills_the_context(dev):
    """A prompt and token budget that use the whole context (n_prompt + new == max_ctx, the runner's
    limit, llm_runner.c:169-173): a ragged last chunk padded to the bucket, the decode steps up to the
    last position the schedule reaches, in the largest bucket, and the oracle's tokens."""
    model, ref = build_pair(synth.TINY, 32, 128)
    prompt = synth.prompt_ids(100, 1024, seed=5)
    want = R.generate(ref, prompt, 28, 16, [64, 128])
    res = llm_runner.run(model, prompt, 28, 16, [64, 128])
    assert res["tokens"] == want
    assert [L for L, _ in res["chunks"]] == [64, 64, 64, 64, 128, 128, 128]
    assert res["decode_steps"] == 27 and {L for L, _ in res["steps"]} == {128}
    with pytest.raises(llm_runner.RunnerError, match="exceeds max_ctx"):
        llm_runner.run(model, prompt, 29, 16, [64, 128])


def test_runner_ragged_prompt_and_stop_ids(dev):
    model, ref = build_pair(synth.TINY, 32, 128)
    prompt = synth.prompt_ids(21, 1024, seed=3)
    want = R.generate(ref, prompt, 10, 8, [16, 32, 64])
    res = llm_runner.run(model, prompt, 10, 8, [16, 32, 64])
    assert res["tokens"] == want
    assert [L for L, _ in res["chunks"]] == [16, 16, 32]
    stop = want[3]
    res2 = llm_runner.run(model, prompt, 10, 8, [16, 32, 64], stop_ids={stop})
    assert res2["tokens"] == want[: want.index(stop) + 1]


def test_runner_multi_step_decode_matches_one_step(dev):
    """Decode replays of 8 steps (one graph, one readback; single steps where a run would cross a
    bucket or the end) give the oracle's tokens across bucket switches, as one-step replays do, and
    their steps read the positions of the caches the one-step run writes."""
    model, ref = build_pair(synth.TINY, 32, 128)
    prompt = synth.prompt_ids(10, 1024, seed=8)
    want = R.generate(ref, prompt, 60, 8, [16, 32, 64, 128])
    c1, c8 = model.new_caches(), model.new_caches()
    one = llm_runner.run(model, prompt, 60, 8, [16, 32, 64, 128], caches=c1, decode_steps=1)
    run8 = llm_runner.run(model, prompt, 60, 8, [16, 32, 64, 128], caches=c8, decode_steps=8)
    assert one["tokens"] == want and run8["tokens"] == want
    for a, b in zip(c1, c8):  # rows 0 .. 68 written, the same values
        assert torch.equal(a[:69], b[:69])


def test_graph_replay_matches_eager_step(dev):
    """The captured entry point, replayed several times with eager work in between, equals step()."""
    model, _ = build_pair(synth.TINY, 32, 128)
    caches_g, caches_e = model.new_caches(), model.new_caches()
    fn = model.entry_point(1, 64, caches_g, logits=True)
    for pos, tok in [(0, 5), (1, 17), (2, 900), (3, 3)]:
        lg = fn([tok], pos, 0).clone()
        _ = torch.randn(1000, device=dev).sum()  # unrelated eager work between replays
        torch.cuda.synchronize()
        _, le = model.step(torch.tensor([[tok]], dtype=torch.int32), torch.tensor([pos], dtype=torch.int32),
                           torch.tensor([0], dtype=torch.int32), caches_e, 64)
        assert torch.equal(lg, le)
    for a, b in zip(caches_g, caches_e):
        assert torch.equal(a, b)


@pytest.mark.parametrize("chunk,buckets", [(256, [256, 512]), (128, [256, 256, 512, 512])])
def test_llama32_3b_generation_matches_golden(dev, chunk, buckets):
    """Llama-3.2-3B shape, synthetic N(0, 0.02) int4 weights (group 128), 512-token
    prompt, 256 greedy tokens over buckets 256..4096: the token ids equal the CPU oracle's
    (tests/golden/make_golden.py 3b, chunks of 256) exactly, prefilled in chunks of 256 (the BASELINE
    config) and of 128 (the reference runner's default, which takes the 128-row prefill kernels).
    Chunks of 64 flip a near tie at token 84 instead: there the two best logits of the oracle's
    sequence are 4.7694 and 4.7693, 1.8e-5 of the largest |logit| apart, and the fp16 K/V rows written
    by a different chunking move them by ~1e-4."""
    gold = json.loads((GOLD / "llama32_3b_tokens.json").read_text())
    sd = synth.PrefetchingWeights(synth.LLAMA32_3B, gold["seed"])
    model = LlamaQ4(None, group=gold["group"], max_ctx=gold["max_ctx"], sd=sd, cfg=synth.LLAMA32_3B)
    sd.close()
    res = llm_runner.run(model, gold["prompt"], gold["max_new_tokens"], chunk, gold["buckets"])
    assert [L for L, _ in res["chunks"]] == buckets
    assert res["tokens"] == gold["tokens"]
    del model
    torch.cuda.empty_cache()


def test_prefill_swiglu_epilogue_matches_two_kernels_and_oracle(dev, kernel_override):
    """A 256-row chunk with intermediate 8192 takes the gate/up GEMM with the SwiGLU epilogue (planes of
    silu(gate) * up written by the GEMM): bit-identical logits and caches to the GEMM + silu_mul pair
    (the swiglu_unfused override), and the oracle's next token with logits within the per-op tolerance."""
    cfg = dict(synth.TINY, intermediate_size=8192, num_hidden_layers=2)
    ours, ref = build_pair(cfg, 32, 256)
    assert ranges(ours, 256, 256)[2] == 0
    prompt = synth.prompt_ids(256, cfg["vocab_size"], seed=3)
    toks = torch.tensor([prompt], dtype=torch.int32)
    start, last = torch.tensor([0], dtype=torch.int32), torch.tensor([255], dtype=torch.int32)
    c_fused = ours.new_caches()
    n_f, l_f = ours.step(toks, start, last, c_fused, 256)
    kernel_override("swiglu_unfused", 1)
    c_two = ours.new_caches()
    n_t, l_t = ours.step(toks, start, last, c_two, 256)
    kernel_override("swiglu_unfused", None)
    assert torch.equal(l_f, l_t) and int(n_f.item()) == int(n_t.item())
    for a, b in zip(c_fused, c_two):
        assert torch.equal(a, b)
    r_n, r_l = ref.step(toks, start, last, ref.new_caches(), 256)
    assert int(n_f.item()) == int(r_n.item())
    assert (l_f.cpu() - r_l).abs().max().item() <= tol(r_l)


def test_prefill_chunk128_k_split_paths_vs_oracle(dev, kernel_override):
    """A 128-row chunk takes every K-split path of the prefill step: qkv, o and down split and completed
    by the RoPE / rms_norm kernels after them, and gate/up (too few 64x256 tiles at 128 rows for its
    SwiGLU epilogue) split too, its partials added by the silu_mul kernel: bit-identical to adding
    them with the reduce kernel first (the swiglu_unfused override). Two chunks (the second reading the first's
    caches), next token and logits against the oracle."""
    cfg = dict(synth.TINY, num_hidden_layers=2, **SPLIT_DIMS)
    ours, ref = build_pair(cfg, 32, 256)
    assert min(ranges(ours, 128, 256)) > 1
    prompt = synth.prompt_ids(256, cfg["vocab_size"], seed=5)
    c_ours, c_two, c_ref = ours.new_caches(), ours.new_caches(), ref.new_caches()
    for s0 in (0, 128):
        toks = torch.tensor([prompt[s0:s0 + 128]], dtype=torch.int32)
        start, last = torch.tensor([s0], dtype=torch.int32), torch.tensor([127], dtype=torch.int32)
        n_o, l_o = ours.step(toks, start, last, c_ours, 256)
        kernel_override("swiglu_unfused", 1)
        n_t, l_t = ours.step(toks, start, last, c_two, 256)
        kernel_override("swiglu_unfused", None)
        assert torch.equal(l_o, l_t) and int(n_o.item()) == int(n_t.item()), s0
        for a, b in zip(c_ours, c_two):
            assert torch.equal(a, b), s0
        r_n, r_l = ref.step(toks, start, last, c_ref, 256)
        assert int(n_o.item()) == int(r_n.item()), s0
        assert (l_o.cpu() - r_l).abs().max().item() <= tol(r_l), s0


@pytest.mark.parametrize("chunk", [2, 15, 16, 17, 32, 33])
@pytest.mark.parametrize("cfg_kw", [dict(), dict(hidden_size=512, intermediate_size=4160), dict(hidden_size=2048)])
def test_prefill_few_rows_vs_oracle(dev, cfg_kw, chunk):
    """Chunks on both sides of the line between the few-rows projections and the tiled ones (16 rows; 32
    rows of dim up to 2048; an inter size past 4096 tiles from 17 rows on): two chunks, the second reading
    the first's caches, next token and logits against the oracle."""
    cfg = dict(synth.TINY, num_hidden_layers=2, **cfg_kw)
    ours, ref = build_pair(cfg, 32, 128)
    prompt = synth.prompt_ids(2 * chunk, cfg["vocab_size"], seed=chunk)
    c_ours, c_ref = ours.new_caches(), ref.new_caches()
    for s0 in (0, chunk):
        toks = torch.tensor([prompt[s0:s0 + chunk]], dtype=torch.int32)
        start, last = torch.tensor([s0], dtype=torch.int32), torch.tensor([chunk - 1], dtype=torch.int32)
        n_o, l_o = ours.step(toks, start, last, c_ours, 128)
        r_n, r_l = ref.step(toks, start, last, c_ref, 128)
        assert int(n_o.item()) == int(r_n.item()), s0
        assert (l_o.cpu() - r_l).abs().max().item() <= tol(r_l), s0


@pytest.mark.parametrize("cfg_kw,chunk,splits", [
    # K ranges of qkv, o, gate/up and down. rms_norm (o, down) loads up to 6 or 12 partials with the row and the
    # rest in a loop; RoPE (qkv) and silu_mul (gate/up) 8, then a loop
    (SPLIT_DIMS, 128, [8, 11, 4, 16]),
    (SPLIT_DIMS, 256, [4, 8, 2, 8]),
    (SPLIT_DIMS, 64, [11, 16, 8, 16]),
    (dict(SPLIT_DIMS, hidden_size=3072, intermediate_size=2048), 256, [4, 5, 4, 5]),
    (dict(SPLIT_DIMS, hidden_size=3072, intermediate_size=2048), 64, [12, 11, 12, 11]),
    # only down splits
    (dict(intermediate_size=8192), 128, [1, 1, 1, 16]),
])
def test_prefill_deferred_partials_bit_identical_to_reduce_kernel(dev, kernel_override, cfg_kw, chunk, splits):
    """The kernels that add a K-split projection's partials themselves (RoPE + KV write after qkv,
    rms_norm after o and down, silu_mul after a split gate/up, the final norm's selected row) give the
    same bits as reducing each projection with linear_reduce_kernel first and running the plain
    kernels (the reduce_splits override): logits, next token and every K/V cache, chunk after chunk."""
    cfg = dict(synth.TINY, num_hidden_layers=2, **cfg_kw)
    ours, ref = build_pair(cfg, 32, 256)
    assert ranges(ours, chunk, 256) == splits
    prompt = synth.prompt_ids(256, cfg["vocab_size"], seed=7)
    c_def, c_red, c_ref = ours.new_caches(), ours.new_caches(), ref.new_caches()
    for s0 in range(0, 256, chunk):
        toks = torch.tensor([prompt[s0:s0 + chunk]], dtype=torch.int32)
        start, last = torch.tensor([s0], dtype=torch.int32), torch.tensor([chunk - 1], dtype=torch.int32)
        n_d, l_d = ours.step(toks, start, last, c_def, 256)
        kernel_override("reduce_splits", 1)
        n_r, l_r = ours.step(toks, start, last, c_red, 256)
        kernel_override("reduce_splits", None)
        assert torch.equal(l_d, l_r) and int(n_d.item()) == int(n_r.item()), s0
        for a, b in zip(c_def, c_red):
            assert torch.equal(a, b), s0
        r_n, r_l = ref.step(toks, start, last, c_ref, 256)
        assert int(n_d.item()) == int(r_n.item()), s0
        assert (l_d.cpu() - r_l).abs().max().item() <= tol(r_l), s0


T16_DIMS = dict(hidden_size=1024, num_attention_heads=8, num_key_value_heads=4, head_dim=128, intermediate_size=8192)


@pytest.mark.parametrize("cfg_kw,group,chunk,tile,plan", [
    # (tile entry, K ranges) of qkv, o, gate/up and down; entries 0 (128x256) and 2 (64x256) read T16
    (T16_DIMS, 128, 256, None, ((1, 1), (2, 8), (2, 0), (2, 16))),  # gate/up: the SwiGLU epilogue
    (T16_DIMS, 128, 128, None, ((2, 8), (2, 8), (2, 2), (2, 16))),
    (dict(T16_DIMS, intermediate_size=1024), 128, 100, None, ((2, 8),) * 4),  # every projection K-split
    (T16_DIMS, 128, 300, None, ((1, 1), (1, 1), (0, 1), (1, 1))),  # more than 256 rows: gate/up on 128x256
    (dict(hidden_size=256, num_attention_heads=64, num_key_value_heads=32, head_dim=128, intermediate_size=4096), 32, 300,
     None, ((0, 1), (1, 1), (1, 1), (1, 1))),  # qkv (RoPE pairing) on 128x256
    # every projection on one of the two tiles
    (T16_DIMS, 128, 300, 0, ((0, 1),) * 4),
    (T16_DIMS, 128, 100, 2, ((2, 1),) * 4),
    (dict(T16_DIMS, intermediate_size=1024), 128, 130, 0, ((0, 1),) * 4),
])
def test_prefill_t16_source_matches_reference_layout(dev, kernel_override, cfg_kw, group, chunk, tile, plan):
    """Prefill projections on the 64x256 and 128x256 tiles read the decode T16 copies (RoPE-paired qkv, plain o
    and down, SwiGLU-paired gate/up) instead of the reference layout: the same sums in the same order, so
    the logits and the K/V caches are bit-identical to the prefill_ref_layout override, and the token matches
    the oracle."""
    cfg = dict(synth.TINY, num_hidden_layers=2, **cfg_kw)
    ours, ref = build_pair(cfg, group, 512)
    kernel_override("linear_tile", tile)
    L = 256 if chunk <= 256 else 512
    assert ours.step_plan(chunk, L) == plan
    assert all((i, nm) in ours.t16 for i in range(2) for nm, (t, _) in zip(("wqkv", "wo", "wgu", "wdown"), plan) if t != 1)
    prompt = synth.prompt_ids(512, cfg["vocab_size"], seed=11)
    toks = torch.tensor([prompt[:chunk]], dtype=torch.int32)
    start, last = torch.tensor([0], dtype=torch.int32), torch.tensor([chunk - 1], dtype=torch.int32)
    c_t = ours.new_caches()
    n_t, l_t = ours.step(toks, start, last, c_t, L)
    kernel_override("prefill_ref_layout", 1)
    c_r = ours.new_caches()
    n_r, l_r = ours.step(toks, start, last, c_r, L)
    kernel_override("prefill_ref_layout", None)
    assert torch.equal(l_t, l_r) and int(n_t.item()) == int(n_r.item())
    for a, b in zip(c_t, c_r):
        assert torch.equal(a, b)
    r_n, r_l = ref.step(toks, start, last, ref.new_caches(), L)
    assert int(n_t.item()) == int(r_n.item())
    assert (l_t.cpu() - r_l).abs().max().item() <= tol(r_l)


def test_prefill_scales_off_a_word_vs_oracle(dev, kernel_override):
    """A model whose group scales start between two words (a C caller's own buffers): the prefill takes the
    kernels that read them one by one; next token and logits against the oracle."""
    ours, ref = build_pair(dict(synth.TINY, num_hidden_layers=2), 32, 128)
    kernel_override("prefill_ref_layout", 1)
    for ly in ours.layers:
        for lin in (ly.wqkv, ly.wo, ly.wgu, ly.wdown):
            buf = torch.empty(lin.scales.numel() + 1, dtype=torch.float16, device=dev)
            buf[1:].copy_(lin.scales.reshape(-1))
            lin.scales = torch.nn.Parameter(buf[1:].view(lin.scales.shape), requires_grad=False)
            assert lin.scales.data_ptr() % 4 == 2
    ours._desc = None
    prompt = synth.prompt_ids(100, 1024, seed=2)
    toks = torch.tensor([prompt], dtype=torch.int32)
    start, last = torch.tensor([0], dtype=torch.int32), torch.tensor([99], dtype=torch.int32)
    n_o, l_o = ours.step(toks, start, last, ours.new_caches(), 128)
    r_n, r_l = ref.step(toks, start, last, ref.new_caches(), 128)
    assert int(n_o.item()) == int(r_n.item())
    assert (l_o.cpu() - r_l).abs().max().item() <= tol(r_l)


def test_group16_step_and_generation_vs_oracle(dev):
    """group 16 (legal in the reference: group % 8 == 0, llama_q4.py:31): the matrix-core prefill GEMM
    takes only groups of 32 * 2^j, so prefill runs one GEMV per row; decode takes the generic GEMV
    path. Logits within the per-op tolerance and greedy tokens equal to the oracle's."""
    ours, ref = build_pair(synth.TINY, 16, 128)
    assert ours.inter == 688
    prompt = synth.prompt_ids(16, 1024, seed=0)
    toks = torch.tensor([prompt], dtype=torch.int32)
    start, last = torch.tensor([0], dtype=torch.int32), torch.tensor([15], dtype=torch.int32)
    n1, l1 = ours.step(toks, start, last, ours.new_caches(), 64)
    r1, rl1 = ref.step(toks, start, last, ref.new_caches(), 64)
    assert int(n1.item()) == int(r1.item())
    assert (l1.cpu() - rl1).abs().max().item() <= tol(rl1)
    want = R.generate(ref, prompt, 12, 8, [16, 32, 64])
    assert llm_runner.run(ours, prompt, 12, 8, [16, 32, 64])["tokens"] == want


def test_no_warmup_entry_points_built_mid_generation(dev):
    """warm-up 0: each entry point is first built after earlier chunks (or the prompt) are in the
    caches, including a prefill bucket switch (16 -> 32) and a decode bucket switch (32 -> 64).
    Building an entry point must leave the live K/V rows intact, so the tokens equal the oracle's."""
    model, ref = build_pair(synth.TINY, 32, 128)
    prompt = synth.prompt_ids(21, 1024, seed=3)
    want = R.generate(ref, prompt, 20, 8, [16, 32, 64])
    res = llm_runner.run(model, prompt, 20, 8, [16, 32, 64], warmup=0)
    assert sorted({L for L, _ in res["steps"]}) == [32, 64]
    assert res["tokens"] == want


def test_step_feed_advances_position_and_matches_step(dev):
    """q4llm_step_feed (include/q4llm.h): the same next token and logits as q4llm_step, and start
    advanced by C on the device by the step's last kernel; tokens == next for a decode step."""
    import ctypes as C
    from q4llm._lib import LIB, ptr, stream_of
    model, _ = build_pair(synth.TINY, 32, 128)
    desc = C.byref(model.descriptor())
    for Cn, pos in ((1, 5), (8, 16)):
        c_a, c_b = model.new_caches(), model.new_caches()
        toks = torch.tensor(synth.prompt_ids(Cn, 1024, seed=pos), dtype=torch.int32, device=dev)
        last = torch.tensor([Cn - 1], dtype=torch.int32, device=dev)
        outs = []
        for feed, caches in ((False, c_a), (True, c_b)):
            start = torch.tensor([pos], dtype=torch.int32, device=dev)
            nxt = torch.empty(1, dtype=torch.int32, device=dev)
            lg = torch.empty(model.embed.vocab, dtype=torch.float32, device=dev)
            ws = model.workspace(Cn, 64)
            LIB.call("q4llm_step_feed" if feed else "q4llm_step", desc, ptr(toks), Cn, ptr(start), ptr(last),
                     model._cache_ptrs(caches), 64, ptr(nxt), ptr(lg), ptr(ws), ws.numel(), stream_of(dev))
            torch.cuda.synchronize()
            outs.append((int(nxt.item()), lg.clone(), int(start.item())))
        assert outs[0][0] == outs[1][0] and torch.equal(outs[0][1], outs[1][1])
        assert outs[0][2] == pos and outs[1][2] == pos + Cn
        for a, b in zip(c_a, c_b):
            assert torch.equal(a, b)

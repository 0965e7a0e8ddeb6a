"""Performance cases of the int4 LLM path: what a program that uses this package has it do.

Each case is a dict of plain values; `prepare` makes what the program holds before the call, `run` is
one pass through the package's public entry points, `exact` is the same result from plain torch in 64
bits, `work` the bytes and operations the pass cannot do without and `tolerance` how far two correct
implementations at the same precision may lie apart.

Kinds:
  gemv      ops.q4_gemv on an fp16 row (the bench's headline call)
  linear    QLinear.forward on fp32 rows: M == 1 is decode, M > 1 a prompt or a batch of rows
  gemm      ops.gemm_f16_nt / gemm_f16_nt_ws, the fp16 NT problems of the gemm harness
  attn      ops.attn_bucket over an fp16 KV bucket: C == 1 decode, C > 1 a prefill chunk
  model     LlamaQ4.entry_point(C, L, logits=True): one captured step that returns its logits
  quantize  quantize_q4 of an fp32 weight (model load)
"""

import importlib
import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "iree-adreno-genai-tuner_amd"))
ops = importlib.import_module("q4llm.ops")
llama = importlib.import_module("q4llm.llama_q4")

DEV = "cuda"
BUCKETS = (256, 512, 1024, 2048, 4096)  # the runner's default KV buckets

# The Llama-3.2-3B shape of the generation benchmark (RoPE without frequency scaling: the tables are data).
MODEL_3B = dict(hidden=3072, layers=28, heads=24, kv=8, hd=128, inter=8192, vocab=128256, group=128)


def listed():
    return [
        # the bench's headline: one fused qkv projection of the 3B shape at decode, fp16 activations
        dict(name="gemv f16 5120x3072", kind="gemv", n=5120, k=3072, group=128),
        # one decode projection through the module API at its default group, with the residual it is added to
        dict(name="linear 1x3072x8192 g32", kind="linear", m=1, n=3072, k=8192, group=32, residual=True),
        # a very short prompt, or a few sequences decoded together
        dict(name="linear 7x3072x3072", kind="linear", m=7, n=3072, k=3072, group=128, residual=True),
        # a ragged prompt at the default group through the widest projection
        dict(name="linear 100x16384x3072 g32", kind="linear", m=100, n=16384, k=3072, group=32, residual=False),
        # a long prompt through the fused qkv projection
        dict(name="linear 512x5120x3072", kind="linear", m=512, n=5120, k=3072, group=128, residual=False),
        # the large square GEMM of the fp16 benchmark
        dict(name="gemm 4096x4096x4096", kind="gemm", m=4096, n=4096, k=4096, ws=False),
        # a ragged prefill chunk through a down projection in fp16, with a workspace
        dict(name="gemm 250x3072x8192 ws", kind="gemm", m=250, n=3072, k=8192, ws=True),
        # decode attention deep in the largest default bucket
        dict(name="attn decode 4096", kind="attn", c=1, heads=24, kv=8, hd=128, l=4096, start=3484),
        # the last prefill chunk of a 2048-token prompt
        dict(name="attn prefill 256 of 2048", kind="attn", c=256, heads=24, kv=8, hd=128, l=2048, start=1792),
        # one decode step of the generation benchmark
        dict(name="3B decode step", kind="model", c=1, l=1024, start=700, **MODEL_3B),
        # its second prefill chunk
        dict(name="3B prefill 256", kind="model", c=256, l=512, start=256, **MODEL_3B),
        # loading a checkpoint: the gate/up weight of one layer
        dict(name="quantize 16384x3072", kind="quantize", n=16384, k=3072, group=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(v, m):
    return max(m, v // m * m)


def draw(rng):
    kind = rng.choice(["gemv", "linear", "linear", "gemm", "attn", "model", "quantize"])
    group = rng.choice([32, 64, 128])
    n, k = _log(rng, 256, 16384), _mult(_log(rng, 256, 8192), max(64, group))
    if kind in ("gemv", "quantize"):
        return dict(kind=kind, n=n, k=k, group=group)
    if kind == "linear":
        m = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 1024)])
        return dict(kind=kind, m=m, n=n, k=k, group=group, residual=rng.random() < 0.5)
    if kind == "gemm":
        m, n, k = _log(rng, 1, 4096), _log(rng, 64, 4096), _mult(_log(rng, 32, 4096), 8)
        return dict(kind=kind, m=m, n=n, k=k, ws=rng.random() < 0.5)
    l = rng.choice(BUCKETS)
    c = rng.choice([1, _log(rng, 2, 256)])
    start = rng.randrange(0, l - c + 1)
    heads, kv, hd = rng.choice([(24, 8, 128), (32, 8, 128), (32, 8, 64), (4, 2, 64), (12, 12, 64), (20, 4, 128)])
    if kind == "attn":
        return dict(kind=kind, c=c, heads=heads, kv=kv, hd=hd, l=l, start=start)
    return dict(kind=kind, c=c, l=l, start=start, hidden=_mult(_log(rng, 256, 3072), 128), layers=rng.randint(1, 4),
                heads=heads, kv=kv, hd=hd, inter=_mult(_log(rng, 512, 8192), 128), vocab=_log(rng, 1000, 32000),
                group=group)


# ------------------------------------------------------------------------------------------------
# Inputs, from the seed alone
# ------------------------------------------------------------------------------------------------


def _normal(seed, index, shape, dtype=torch.float32, std=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + index)
    return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, std, generator=g).to(dtype)


def _weight(case, seed):
    return _normal(seed, 1, (case["n"], case["k"]), std=0.02)


class _Checkpoint:
    """State dict of a random Llama, its tensors made when they are asked for."""

    def __init__(self, case, seed):
        c, self.seed = case, seed
        h, nq, nkv, inter = c["hidden"], c["heads"] * c["hd"], c["kv"] * c["hd"], c["inter"]
        shapes = {"model.embed_tokens.weight": (c["vocab"], h), "model.norm.weight": (h,)}
        for i in range(c["layers"]):
            p = f"model.layers.{i}."
            shapes.update({p + "self_attn.q_proj.weight": (nq, h), p + "self_attn.k_proj.weight": (nkv, h),
                           p + "self_attn.v_proj.weight": (nkv, h), p + "self_attn.o_proj.weight": (h, nq),
                           p + "mlp.gate_proj.weight": (inter, h), p + "mlp.up_proj.weight": (inter, h),
                           p + "mlp.down_proj.weight": (h, inter), p + "input_layernorm.weight": (h,),
                           p + "post_attention_layernorm.weight": (h,)})
        self.shapes = {name: (10 + i, s) for i, (name, s) in enumerate(shapes.items())}

    def __contains__(self, name):
        return name in self.shapes

    def __getitem__(self, name):
        i, shape = self.shapes[name]
        if len(shape) == 1:
            return 1.0 + _normal(self.seed, i, shape, std=0.1)
        return _normal(self.seed, i, shape, std=0.02)


def _tokens(case, seed):
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randint(0, case["vocab"], (case["c"],), generator=g, dtype=torch.int32)


def _past(case, seed, index):
    """A cache [l, kv, hd] with the rows before `start` filled, as a running generation leaves it."""
    t = _normal(seed, index, (case["l"], case["kv"], case["hd"]), torch.float16)
    t[case["start"]:] = 0
    return t


def _attn_inputs(case, seed):
    """The fused qkv rows and the caches with this chunk's K and V rows written."""
    c, nq, nkv = case["c"], case["heads"] * case["hd"], case["kv"] * case["hd"]
    qkv = _normal(seed, 1, (c, nq + 2 * nkv))
    kc, vc = _past(case, seed, 2), _past(case, seed, 3)
    s = case["start"]
    kc[s:s + c] = qkv[:, nq:nq + nkv].reshape(c, case["kv"], case["hd"]).half()
    vc[s:s + c] = qkv[:, nq + nkv:].reshape(c, case["kv"], case["hd"]).half()
    return qkv, kc, vc


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        qw, sc = ops.quantize_q4(_weight(case, seed), case["group"])
        return dict(case=case, qw=qw, sc=sc, x=_normal(seed, 2, (case["k"],), torch.float16))
    if kind == "linear":
        res = _normal(seed, 3, (case["m"], case["n"])) if case["residual"] else None
        return dict(case=case, mod=llama.QLinear(_weight(case, seed), case["group"]),
                    x=_normal(seed, 2, (case["m"], case["k"])), res=res)
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        ws = None
        if case["ws"]:
            ws = torch.empty(max(16, ops.gemm_f16_nt_ws_bytes(m, n, k)), dtype=torch.uint8, device=DEV)
        return dict(case=case, a=_normal(seed, 1, (m, k), torch.float16), b=_normal(seed, 2, (n, k), torch.float16),
                    ws=ws)
    if kind == "attn":
        qkv, kc, vc = _attn_inputs(case, seed)
        q = qkv[:, :case["heads"] * case["hd"]].unflatten(1, (case["heads"], case["hd"]))
        nbytes = ops.attn_workspace_bytes(case["c"], case["heads"], case["kv"], case["hd"], case["l"])
        return dict(case=case, q=q, kc=kc, vc=vc, start=torch.full((1,), case["start"], dtype=torch.int32, device=DEV),
                    ws=torch.empty(max(1, nbytes), dtype=torch.uint8, device=DEV))
    if kind == "model":
        cfg = dict(hidden_size=case["hidden"], num_hidden_layers=case["layers"], num_attention_heads=case["heads"],
                   num_key_value_heads=case["kv"], head_dim=case["hd"], intermediate_size=case["inter"],
                   vocab_size=case["vocab"], rms_norm_eps=1e-5, rope_theta=500000.0, tie_word_embeddings=True)
        model = llama.LlamaQ4(group=case["group"], max_ctx=case["l"], sd=_Checkpoint(case, seed), cfg=cfg)
        caches = [_past(case, seed, 1000 + i) for i in range(2 * case["layers"])]
        fn = model.entry_point(case["c"], case["l"], caches, logits=True)
        return dict(case=case, model=model, caches=caches, fn=fn, tokens=_tokens(case, seed))
    return dict(case=case, w=_weight(case, seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        return ops.q4_gemv(state["qw"], state["sc"], state["x"], case["group"], out_dtype=torch.float16)
    if kind == "linear":
        return state["mod"](state["x"], residual=state["res"])
    if kind == "gemm":
        if case["ws"]:
            return ops.gemm_f16_nt_ws(state["a"], state["b"], workspace=state["ws"])
        return ops.gemm_f16_nt(state["a"], state["b"])
    if kind == "attn":
        return ops.attn_bucket(state["q"], state["kc"], state["vc"], case["l"], state["start"],
                               1.0 / math.sqrt(case["hd"]), workspace=state["ws"])
    if kind == "model":
        logits = state["fn"](state["tokens"], case["start"], case["c"] - 1)
        return dict(logits=logits, caches=state["caches"])
    return llama.quantize_q4(state["w"], case["group"])


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------------------


def _weight_bytes(n, k, group):
    return n * k / 2 + n * (k // group) * 2


def _valid(case):
    """Keys that the chunk's rows attend to, summed over the rows."""
    return sum(case["start"] + i + 1 for i in range(case["c"]))


def _attn_work(case):
    c, nq, nkv = case["c"], case["heads"] * case["hd"], case["kv"] * case["hd"]
    return (case["start"] + c) * nkv * 4 + c * nq * 8, 4 * _valid(case) * nq


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n, k = case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, case["group"]) + 2 * k + 2 * n, "flops": 2 * n * k}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, case["group"]) + 4 * m * k + 4 * m * n * (2 if case["residual"] else 1),
                "flops": 2 * m * n * k}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "attn":
        b, f = _attn_work(case)
        return {"bytes": b, "flops": f}
    if kind == "model":
        c, h, g, inter = case["c"], case["hidden"], case["group"], case["inter"]
        nq, nkv = case["heads"] * case["hd"], case["kv"] * case["hd"]
        shapes = [(nq + 2 * nkv, h), (h, nq), (2 * inter, h), (h, inter)]
        per_layer = sum(_weight_bytes(n, k, g) for n, k in shapes) + (case["start"] + 2 * c) * nkv * 4
        flops = case["layers"] * (sum(2 * c * n * k for n, k in shapes) + _attn_work(case)[1]) + 2 * case["vocab"] * h
        return {"bytes": case["layers"] * per_layer + _weight_bytes(case["vocab"], h, g) + 4 * case["vocab"],
                "flops": flops}
    n, k = case["n"], case["k"]
    return {"bytes": 4 * n * k + _weight_bytes(n, k, case["group"]), "flops": 4 * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"  # integers, and scales of one fp32 division rounded once to fp16
    # about four times the largest error against 64 bits seen over the listed and fourteen drawn cases
    if kind in ("gemv", "gemm"):
        return {"rel": 8e-4, "max": 2e-3}  # one fp16 rounding of the result each
    if kind in ("linear", "attn"):
        return {"rel": 1.2e-6, "max": 1.2e-5}  # fp32 products, softmax and sums
    return {"rel": 5e-4, "max": 4e-3}  # fp32 activations; K and V rows are rounded to fp16 in every layer


# ------------------------------------------------------------------------------------------------
# The same results in 64 bits
# ------------------------------------------------------------------------------------------------


def _quantized(w, group):
    """(integers in [-8, 7], fp16 scales) of the int4 format."""
    n, k = w.shape
    g = w.reshape(n, k // group, group)
    amax = g.abs().amax(-1, keepdim=True).clamp_min(1e-8)
    scale = amax / torch.full_like(amax, 7.0)  # by a tensor: a true division, not a product with 1 / 7
    return torch.clamp(torch.round(g / scale), -8, 7), scale.squeeze(-1).half()


def _dequant64(w, group):
    q, s = _quantized(w, group)
    return (q.double() * s.double().unsqueeze(-1)).reshape(w.shape)


def _attend64(q, kc, vc, start):
    """q [C, heads, hd], caches [L, kv, hd], all fp64 -> [C, heads * hd]."""
    c, heads, hd = q.shape
    n, kv = start + c, kc.shape[1]
    pos = torch.arange(start, start + c, device=q.device)
    mask = torch.arange(n, device=q.device)[None, :] > pos[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        j = h // (heads // kv)
        s = q[:, h].contiguous() @ kc[:n, j].contiguous().t().contiguous() / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ vc[:n, j].contiguous()
    return out.reshape(c, heads * hd)


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w


def _rotate64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos[:, None] + torch.cat((-x[..., half:], x[..., :half]), -1) * sin[:, None]


def _model64(case, seed):
    sd, g, c, s = _Checkpoint(case, seed), case["group"], case["c"], case["start"]
    heads, kv, hd, inter = case["heads"], case["kv"], case["hd"], case["inter"]
    nq, nkv = heads * hd, kv * hd
    inv = 1.0 / (500000.0 ** (torch.arange(0, hd, 2).float() / hd))
    ang = torch.arange(s, s + c).float()[:, None] * inv[None, :]  # the tables are fp32 products
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos().double().to(DEV), ang.sin().double().to(DEV)
    embed = sd["model.embed_tokens.weight"]
    h = _dequant64(embed[_tokens(case, seed).long().to(DEV)], g)
    caches = []
    for i in range(case["layers"]):
        p = f"model.layers.{i}."

        def linear(x, name):
            return x @ _dequant64(sd[p + name + ".weight"], g).t()

        x = _norm64(h, sd[p + "input_layernorm.weight"].double())
        q = _rotate64(linear(x, "self_attn.q_proj").reshape(c, heads, hd), cos, sin)
        k = _rotate64(linear(x, "self_attn.k_proj").reshape(c, kv, hd), cos, sin)
        v = linear(x, "self_attn.v_proj").reshape(c, kv, hd)
        kc, vc = _past(case, seed, 1000 + 2 * i).double(), _past(case, seed, 1001 + 2 * i).double()
        kc[s:s + c], vc[s:s + c] = k.half().double(), v.half().double()
        caches += [kc, vc]
        h = h + linear(_attend64(q, kc, vc, s), "self_attn.o_proj")
        x = _norm64(h, sd[p + "post_attention_layernorm.weight"].double())
        h = h + linear(torch.nn.functional.silu(linear(x, "mlp.gate_proj")) * linear(x, "mlp.up_proj"), "mlp.down_proj")
    x = _norm64(h[c - 1:], sd["model.norm.weight"].double())
    logits = torch.cat([x @ _dequant64(rows, g).t() for rows in embed.split(16384)], -1)
    return dict(logits=logits, caches=caches)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        return _dequant64(_weight(case, seed), case["group"]) @ _normal(seed, 2, (case["k"],), torch.float16).double()
    if kind == "linear":
        y = _normal(seed, 2, (case["m"], case["k"])).double() @ _dequant64(_weight(case, seed), case["group"]).t()
        return y + _normal(seed, 3, (case["m"], case["n"])).double() if case["residual"] else y
    if kind == "gemm":
        a = _normal(seed, 1, (case["m"], case["k"]), torch.float16).double()
        return a @ _normal(seed, 2, (case["n"], case["k"]), torch.float16).double().t()
    if kind == "attn":
        qkv, kc, vc = _attn_inputs(case, seed)
        nq = case["heads"] * case["hd"]
        q = qkv[:, :nq].reshape(case["c"], case["heads"], case["hd"]).double()
        return _attend64(q, kc.double(), vc.double(), case["start"])
    if kind == "model":
        return _model64(case, seed)
    return [None, _quantized(_weight(case, seed), case["group"])[1].double()]

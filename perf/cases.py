"""The work that a user of this engine has it do, as cases that can be timed.

Every case goes through the entry points that a serving program calls: attention
(``flash_attention``, ``flash_decode``), the W8A16 transformer block and its
feed-forward half, the hipGraph decode step of the whole W8A16 model, and the
weight quantiser that a checkpoint passes through at load time.  Two model
shapes occur, the ones the benchmark names:

  1b  dim 2048, 32 query / 8 KV heads, head_dim 64,  FFN 8192, 16 layers
  3b  dim 3072, 24 query / 8 KV heads, head_dim 128, FFN 8192

Kinds and the ranges they stand for (``draw`` samples them):

  prefill        causal GQA attention over a prompt: 1..8 prompts of 32..8192
                 tokens (odd lengths too), bf16 or fp16, q/k/v contiguous with
                 the LSE returned, or in the model's layout (views of
                 [B, S, H, D] projections, K/V in the cache, RoPE(q) fused);
                 fp32 up to 1024 tokens.
  decode         one query token per sequence against a KV cache: 1..16
                 sequences, 64..131072 keys, all keys, per-sequence lengths or
                 a bool mask (left-padded batch).
  block_prefill  one W8A16 transformer block over a prompt (32..8192 rows).
  block_decode   the same block on one token for 1..16 sequences.
  ffn            norm + SwiGLU feed-forward + residual of that block on
                 1..8192 rows (a decode batch, a chat prompt, a long prompt).
  step           a whole decode step through the hipGraph runner.
  quantize       a bf16 weight matrix to int8 with per-channel scales.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "llm-infer-engine_amd"))

from src.config import ModelArgs  # noqa: E402
from src.cuda_graph import CUDAGraphDecodeRunner  # noqa: E402
from src.flash_attn import flash_attention  # noqa: E402
from src.flash_decode import flash_decode  # noqa: E402
from src.kv_cache import KVCache  # noqa: E402
from src.model_quantized import Llama3Quantized, QuantizedTransformerBlock  # noqa: E402
from src.quant_utils import quantize_weight_symmetric_per_channel  # noqa: E402

DEV = "cuda:0"
THETA = 500000.0
EPS = 1e-5
VOCAB = 128256
SHAPES = {  # dim, FFN, query heads, KV heads, head_dim
    "1b": (2048, 8192, 32, 8, 64),
    "3b": (3072, 8192, 24, 8, 128),
}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
LINEARS = ("attention.wq", "attention.wk", "attention.wv", "attention.wo",
           "feed_forward.w1", "feed_forward.w2", "feed_forward.w3")


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # a single user's chat: one token per step, short context
        {"name": "step_chat", "kind": "step", "batch": 1, "ctx": 777, "capacity": 2048},
        # the engine's headline decode step: 8 sequences, 4096 tokens of context
        {"name": "step_batch", "kind": "step", "batch": 8, "ctx": 4096, "capacity": 8192},
        # one layer of a 16-way decode batch of the 3B shape, called eagerly
        {"name": "block_decode", "kind": "block_decode", "shape": "3b", "batch": 16,
         "ctx": 2047, "capacity": 4096},
        # a chat prompt through the feed-forward half of a block
        {"name": "ffn_prompt", "kind": "ffn", "shape": "1b", "rows": 300},
        # the same for a few tokens per call: a large decode batch
        {"name": "ffn_rows", "kind": "ffn", "shape": "3b", "rows": 48},
        # one layer of a batched prefill, the largest call
        {"name": "block_prefill", "kind": "block_prefill", "shape": "1b", "batch": 4,
         "seq": 2048, "capacity": 4096},
        # the headline prefill attention
        {"name": "prefill_batch", "kind": "prefill", "shape": "1b", "batch": 4, "seq": 2048,
         "dtype": "bf16", "layout": "plain"},
        # one document of odd length, as the model calls it
        {"name": "prefill_document", "kind": "prefill", "shape": "3b", "batch": 1, "seq": 3001,
         "dtype": "bf16", "layout": "model"},
        # the fp32 check configuration: one prompt of 512 tokens
        {"name": "prefill_fp32", "kind": "prefill", "shape": "1b", "batch": 1, "seq": 512,
         "dtype": "fp32", "layout": "plain"},
        # continuous batching: 16 sequences of 1024..8192 keys
        {"name": "decode_ragged", "kind": "decode", "shape": "3b", "batch": 16, "keys": 8192,
         "dtype": "bf16", "select": "lengths"},
        # one sequence with a 128 K context
        {"name": "decode_long", "kind": "decode", "shape": "3b", "batch": 1, "keys": 131072,
         "dtype": "bf16", "select": "all"},
        # loading a checkpoint: the largest projection of a layer
        {"name": "quantize", "kind": "quantize", "rows": 8192, "cols": 2048, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "decode", "decode", "decode",
                       "block_prefill", "block_prefill", "block_decode", "block_decode",
                       "ffn", "ffn", "step", "quantize"])
    shape = rng.choice(["1b", "3b"])
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"])
        seq = _log(rng, 32, 1024 if dtype == "fp32" else 8192)
        # at most the attention of 4 prompts of 2048 tokens (fp32: of one of 1024)
        most = max(1, int((1.0 if dtype == "fp32" else 16.0) * 1024 ** 2 / seq ** 2))
        return {"kind": kind, "shape": shape, "batch": rng.randint(1, min(8, most)), "seq": seq,
                "dtype": dtype, "layout": "plain" if dtype == "fp32" else rng.choice(["plain", "model"])}
    if kind == "decode":
        keys = _log(rng, 64, 131072)
        return {"kind": kind, "shape": shape, "batch": rng.randint(1, max(1, min(16, 131072 // keys))),
                "keys": keys, "dtype": rng.choice(["bf16", "bf16", "fp16"]),
                "select": rng.choice(["all", "lengths", "mask"])}
    if kind == "block_prefill":
        seq = _log(rng, 32, 4096)
        batch = rng.randint(1, max(1, min(8, 4096 // seq)))
        return {"kind": kind, "shape": shape, "batch": batch, "seq": seq, "capacity": 4096}
    if kind == "block_decode":
        return {"kind": kind, "shape": shape, "batch": rng.randint(1, 16),
                "ctx": _log(rng, 16, 4095), "capacity": 4096}
    if kind == "ffn":
        return {"kind": kind, "shape": shape, "rows": _log(rng, 1, 8192 if shape == "1b" else 4096)}
    if kind == "step":
        return {"kind": kind, "batch": rng.randint(1, 8), "ctx": _log(rng, 16, 4096), "capacity": 8192}
    return {"kind": kind, "rows": _log(rng, 256, 8192), "cols": 16 * _log(rng, 32, 512),
            "dtype": rng.choice(["bf16", "bf16", "fp16"])}


# ------------------------------------------------------- inputs from the seed

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *size, dtype=torch.bfloat16):
    return torch.randn(size, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _weight(g, n, k):
    """int8 rows of a normal weight matrix (largest value of a row ~4 sigma) and
    scales that keep a product of unit-variance rows at unit variance."""
    q = (torch.randn((n, k), generator=g, device=DEV) * 32.0).round_().clamp_(-127, 127).to(torch.int8)
    s = (torch.rand((n, 1), generator=g, device=DEV) * 0.2 + 0.9) / (32.0 * math.sqrt(k))
    return q, s.to(torch.bfloat16)


def _layer(g, shape):
    dim, hidden, hq, hkv, d = SHAPES[shape]
    sizes = {"attention.wq": (hq * d, dim), "attention.wk": (hkv * d, dim), "attention.wv": (hkv * d, dim),
             "attention.wo": (dim, hq * d), "feed_forward.w1": (hidden, dim),
             "feed_forward.w2": (dim, hidden), "feed_forward.w3": (hidden, dim)}
    w = {name: _weight(g, *sizes[name]) for name in LINEARS}
    w["attention_norm"] = (1.0 + 0.1 * _randn(g, dim, dtype=torch.float32)).to(torch.bfloat16)
    w["ffn_norm"] = (1.0 + 0.1 * _randn(g, dim, dtype=torch.float32)).to(torch.bfloat16)
    return w


def _tables(d, rows, dtype):
    """cos/sin [rows, d/2] in the activation dtype (fp32 angles on the CPU)."""
    f = 1.0 / (THETA ** (torch.arange(0, d, 2).float() / d))
    a = torch.outer(torch.arange(rows), f).float()
    z = torch.polar(torch.ones_like(a), a)
    return z.real.to(device=DEV, dtype=dtype), z.imag.to(device=DEV, dtype=dtype)


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "prefill":
        _, _, hq, hkv, d = SHAPES[case["shape"]]
        b, s, dt = case["batch"], case["seq"], DTYPES[case["dtype"]]
        if case["layout"] == "plain":
            return {"q": _randn(g, b, hq, s, d, dtype=dt), "k": _randn(g, b, hkv, s, d, dtype=dt),
                    "v": _randn(g, b, hkv, s, d, dtype=dt)}
        cap = -(-(s + 256) // 256) * 256   # the cache holds more slots than the prompt fills
        k, v = (_randn(g, b, hkv, cap, d, dtype=dt) for _ in range(2))
        cos, sin = _tables(d, s, dt)
        return {"q": _randn(g, b, s, hq, d, dtype=dt).transpose(1, 2), "k": k[:, :, :s], "v": v[:, :, :s],
                "cos": cos, "sin": sin}
    if kind == "decode":
        _, _, hq, hkv, d = SHAPES[case["shape"]]
        b, n, dt = case["batch"], case["keys"], DTYPES[case["dtype"]]
        t = {"q": _randn(g, b, hq, 1, d, dtype=dt), "k": _randn(g, b, hkv, n, d, dtype=dt),
             "v": _randn(g, b, hkv, n, d, dtype=dt)}
        lens = torch.randint(max(1, n // 8), n + 1, (b,), generator=torch.Generator().manual_seed(int(seed)))
        if case["select"] == "lengths":
            t["lens"] = lens.to(DEV)
        elif case["select"] == "mask":    # left-padded prompts: the last lens[b] keys are visible
            t["mask"] = (torch.arange(n)[None] >= n - lens[:, None]).view(b, 1, 1, n).to(DEV)
        return t
    if kind == "quantize":
        w = _randn(g, case["rows"], case["cols"], dtype=torch.float32) * (1.0 / math.sqrt(case["cols"]))
        return {"w": w.to(DTYPES[case["dtype"]])}
    if kind == "ffn":
        return {"layers": [_layer(g, case["shape"])], "x": _randn(g, case["rows"], SHAPES[case["shape"]][0])}
    if kind in ("block_prefill", "block_decode"):
        dim, _, _, hkv, d = SHAPES[case["shape"]]
        b, cap = case["batch"], case["capacity"]
        t = {"layers": [_layer(g, case["shape"])]}
        t["x"] = _randn(g, b, case["seq"] if kind == "block_prefill" else 1, dim)
        t["cache"] = torch.zeros((2, 1, b, hkv, cap, d), device=DEV, dtype=torch.bfloat16)
        if kind == "block_decode":
            t["cache"][..., :case["ctx"], :] = _randn(g, 2, 1, b, hkv, case["ctx"], d)
        t["cos"], t["sin"] = _tables(d, cap, torch.bfloat16)
        return t
    b, cap, ctx = case["batch"], case["capacity"], case["ctx"]
    dim, _, _, hkv, d = SHAPES["1b"]
    t = {"layers": [_layer(g, "1b") for _ in range(16)], "emb": _randn(g, VOCAB, dim),
         "norm": (1.0 + 0.1 * _randn(g, dim, dtype=torch.float32)).to(torch.bfloat16),
         "out": (_randn(g, VOCAB, dim, dtype=torch.float32) / math.sqrt(dim)).to(torch.bfloat16),
         "tokens": torch.randint(0, VOCAB, (b, 1), generator=g, device=DEV),
         "cache": torch.zeros((2, 16, b, hkv, cap, d), device=DEV, dtype=torch.bfloat16)}
    for kv in t["cache"]:
        for layer in kv:
            layer[:, :, :ctx] = _randn(g, b, hkv, ctx, d)
    return t


# ------------------------------------------------ what the program has in hand

def _args(shape, layers, batch, capacity):
    dim, hidden, hq, hkv, _ = SHAPES[shape]
    return ModelArgs(dim=dim, n_layers=layers, n_heads=hq, n_kv_heads=hkv, vocab_size=VOCAB,
                     hidden_dim=hidden, norm_eps=EPS, max_batch_size=batch, max_seq_len=capacity,
                     rope_theta=THETA, device=DEV)


def _load_block(block, w):
    for name in LINEARS:
        lin = block.get_submodule(name)
        lin.weight.data, lin.scales.data = w[name]
    block.attention_norm.weight.data = w["attention_norm"]
    block.ffn_norm.weight.data = w["ffn_norm"]
    return block.eval()


def _fill(kv, data):
    kv.k.copy_(data[0])
    kv.v.copy_(data[1])


@torch.no_grad()
def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    s = {"kind": kind, "case": case, "t": t}
    if kind in ("ffn", "block_prefill", "block_decode"):
        args = _args(case["shape"], 1, case.get("batch", 1), case.get("capacity", 256))
        with torch.device("meta"):
            block = QuantizedTransformerBlock(args)
        s["block"] = _load_block(block.to_empty(device=DEV), t["layers"][0])
        if kind != "ffn":
            s["kv"] = KVCache(args, dtype=torch.bfloat16)
            _fill(s["kv"], t.pop("cache"))
            at = 0 if kind == "block_prefill" else case["ctx"]
            n = t["x"].shape[1]
            s["rope"] = (t["cos"][at:at + n], t["sin"][at:at + n])
    elif kind == "step":
        args = _args("1b", 16, case["batch"], case["capacity"])
        with torch.device("meta"):
            model = Llama3Quantized(args)
        model = model.to_empty(device=DEV)
        for layer, w in zip(model.layers, t["layers"]):
            _load_block(layer, w)
        model.tok_embeddings.weight.data = t["emb"]
        model.norm.weight.data = t["norm"]
        model.output.weight.data = t["out"]
        # the runner's warm-up writes slot 0: a program captures first, then prefills
        s["kv"] = KVCache(args, dtype=torch.bfloat16)
        s["runner"] = CUDAGraphDecodeRunner(model.eval(), args, s["kv"], DEV, batch_size=case["batch"])
        _fill(s["kv"], t.pop("cache"))
    return s


# ---------------------------------------------------------------- one pass

@torch.no_grad()
def run(s):
    t, kind, case = s["t"], s["kind"], s["case"]
    if kind == "prefill":
        if case["layout"] == "plain":
            return flash_attention(t["q"], t["k"], t["v"], return_lse=True)
        return flash_attention(t["q"], t["k"], t["v"], rope_cos=t["cos"], rope_sin=t["sin"])
    if kind == "decode":
        return flash_decode(t["q"], t["k"], t["v"], t.get("mask"), seq_lens=t.get("lens"))
    if kind == "ffn":
        return s["block"].feed_forward(s["block"].ffn_norm(t["x"]), residual=t["x"])
    if kind in ("block_prefill", "block_decode"):
        at = 0 if kind == "block_prefill" else case["ctx"]
        y = s["block"](t["x"], *s["rope"], layer_idx=0, start_pos=at, kv_cache=s["kv"])
        return {"y": y, "k": s["kv"].k, "v": s["kv"].v}
    if kind == "step":
        logits = s["runner"].decode(t["tokens"], case["ctx"])
        return {"logits": logits, "k": s["kv"].k, "v": s["kv"].v}
    return quantize_weight_symmetric_per_channel(t["w"])


# ------------------------------------------------------ what a pass must move

def _layer_work(shape, rows, parts=LINEARS):
    dim, hidden, hq, hkv, d = SHAPES[shape]
    n = {"attention.wq": hq * d * dim, "attention.wk": hkv * d * dim, "attention.wv": hkv * d * dim,
         "attention.wo": dim * hq * d, "feed_forward.w1": dim * hidden, "feed_forward.w2": dim * hidden,
         "feed_forward.w3": dim * hidden}
    w = sum(n[p] for p in parts)
    return w, 2 * rows * w    # int8 bytes, flops


def work(case):
    kind = case["kind"]
    if kind == "prefill":
        _, _, hq, hkv, d = SHAPES[case["shape"]]
        b, s, es = case["batch"], case["seq"], 4 if case["dtype"] == "fp32" else 2
        lse = 4 * b * hq * s if case["layout"] == "plain" else 0
        return {"bytes": es * b * s * d * (2 * hq + 2 * hkv) + lse, "flops": 4 * b * hq * d * s * (s + 1) // 2}
    if kind == "decode":
        _, _, hq, hkv, d = SHAPES[case["shape"]]
        b, n = case["batch"], case["keys"]
        if case["select"] != "all":    # lengths are uniform in [keys / 8, keys]
            n = (max(1, n // 8) + n) // 2
        return {"bytes": 2 * b * (2 * hkv * n * d + 2 * hq * d), "flops": 4 * b * hq * n * d}
    if kind == "quantize":
        n = case["rows"] * case["cols"]
        return {"bytes": 3 * n + 2 * case["rows"], "flops": 2 * n}
    if kind == "ffn":
        by, fl = _layer_work(case["shape"], case["rows"], LINEARS[4:])
        return {"bytes": by + 4 * case["rows"] * SHAPES[case["shape"]][0], "flops": fl}
    if kind in ("block_prefill", "block_decode"):
        dim, _, hq, hkv, d = SHAPES[case["shape"]]
        b = case["batch"]
        s = case["seq"] if kind == "block_prefill" else 1
        by, fl = _layer_work(case["shape"], b * s)
        by += 4 * b * s * dim + 4 * b * hkv * s * d
        if kind == "block_prefill":
            return {"bytes": by, "flops": fl + 4 * b * hq * d * s * (s + 1) // 2}
        return {"bytes": by + 4 * b * hkv * case["ctx"] * d, "flops": fl + 4 * b * hq * d * (case["ctx"] + 1)}
    dim, _, hq, hkv, d = SHAPES["1b"]
    b, n = case["batch"], case["ctx"] + 1
    by, fl = _layer_work("1b", b)
    return {"bytes": 16 * (by + 4 * b * hkv * n * d) + 2 * VOCAB * dim + 2 * b * VOCAB,
            "flops": 16 * (fl + 4 * b * hq * d * n) + 2 * b * VOCAB * dim}


# ------------------------------------------------------- tolerances and truth

def tolerance(case):
    """About four times the error of the present code against 64 bits: 2e-7 for
    fp32 attention, 2.1e-3 .. 2.5e-3 in bf16 and 2.6e-4 in fp16, 3.0e-3 .. 3.8e-3
    for a bf16 block; 16 layers of bf16 roundings leave 1.6e-2 .. 1.9e-2."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "prefill" and case["dtype"] == "fp32":
        return {"rel": 1e-6}
    if kind in ("prefill", "decode"):
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.2e-3, "max": 0.1}
    if kind == "step":
        return {"rel": 3e-2, "max": 0.3}
    return {"rel": 1.5e-2, "max": 0.1}


def _rope64(x, cos, sin):
    h = x.shape[-1] // 2
    a, b, c, s = x[..., :h], x[..., h:], cos.double(), sin.double()
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _lin64(x, w):
    return (x @ w[0].double().t()) * w[1].double().view(-1)


def _causal64(q, k, v):
    """out, lse of causal attention in 64 bits: q [B, Hq, S, D], k/v [B, Hkv, S, D]."""
    b, hq, n, d = q.shape
    per = hq // k.shape[1]
    out = torch.empty((b, hq, n, d), dtype=torch.float64, device=DEV)
    lse = torch.empty((b, hq, n), dtype=torch.float64, device=DEV)
    hide = torch.ones((n, n), dtype=torch.bool, device=DEV).triu_(1)
    for i in range(b):
        for h in range(hq):
            p = q[i, h].double() @ k[i, h // per].double().t()
            p.mul_(1.0 / math.sqrt(d)).masked_fill_(hide, -math.inf)
            lse[i, h] = torch.logsumexp(p, -1)
            out[i, h] = p.sub_(lse[i, h][:, None]).exp_() @ v[i, h // per].double()
    return out, lse


def _decode64(q, k, v, seen):
    """q [B, Hq, 1, D] over the keys that seen [B, L] selects."""
    b, hq, _, d = q.shape
    per = hq // k.shape[1]
    out = torch.empty((b, hq, 1, d), dtype=torch.float64, device=DEV)
    for i in range(b):
        for h in range(k.shape[1]):
            rows = slice(h * per, (h + 1) * per)
            p = q[i, rows, 0].double() @ k[i, h].double().t() * (1.0 / math.sqrt(d))
            p = torch.softmax(p.masked_fill(~seen[i], -math.inf), -1)
            out[i, rows, 0] = p @ v[i, h].double()
    return out


def _ffn64(x, w):
    h = _norm64(x, w["ffn_norm"])
    g = torch.nn.functional.silu(_lin64(h, w["feed_forward.w1"])) * _lin64(h, w["feed_forward.w3"])
    return x + _lin64(g, w["feed_forward.w2"])


def _block64(x, w, shape, cos, sin, ck, cv, at):
    """x [B, S, dim] at positions at..; ck/cv [B, Hkv, T, D] in 64 bits get the new rows."""
    _, _, hq, hkv, d = SHAPES[shape]
    b, n, _ = x.shape
    h = _norm64(x, w["attention_norm"])
    q, k, v = (_lin64(h, w["attention." + p]).view(b, n, -1, d).transpose(1, 2) for p in ("wq", "wk", "wv"))
    q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
    ck[:, :, at:at + n], cv[:, :, at:at + n] = k, v
    if n > 1:
        o = _causal64(q, k, v)[0]
    else:
        seen = torch.ones((b, at + 1), dtype=torch.bool, device=DEV)
        o = _decode64(q, ck[:, :, :at + 1], cv[:, :, :at + 1], seen)
    return _ffn64(x + _lin64(o.transpose(1, 2).reshape(b, n, -1), w["attention.wo"]), w)


@torch.no_grad()
def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "prefill":
        q = t["q"].double()
        if case["layout"] == "model":
            return _causal64(_rope64(q, t["cos"], t["sin"]), t["k"], t["v"])[0]
        return _causal64(q, t["k"], t["v"])
    if kind == "decode":
        b, n = case["batch"], case["keys"]
        seen = torch.ones((b, n), dtype=torch.bool, device=DEV)
        if "lens" in t:
            seen = torch.arange(n, device=DEV)[None] < t["lens"][:, None]
        elif "mask" in t:
            seen = t["mask"].view(b, n)
        return _decode64(t["q"], t["k"], t["v"], seen)
    if kind == "quantize":
        amax = t["w"].double().abs().amax(1, keepdim=True).clamp_min(1e-12)
        return None, amax / 127.0
    if kind == "ffn":
        return _ffn64(t["x"].double(), t["layers"][0])
    if kind in ("block_prefill", "block_decode"):
        at = 0 if kind == "block_prefill" else case["ctx"]
        n = t["x"].shape[1]
        ck, cv = t["cache"][0, 0].double(), t["cache"][1, 0].double()
        y = _block64(t["x"].double(), t["layers"][0], case["shape"], t["cos"][at:at + n],
                     t["sin"][at:at + n], ck, cv, at)
        return {"y": y, "k": ck[None], "v": cv[None]}
    ctx = case["ctx"]
    cos, sin = _tables(64, ctx + 1, torch.bfloat16)
    x = t["emb"][t["tokens"]].double()
    k, v = t["cache"].double().unbind(0)
    for i, w in enumerate(t["layers"]):
        x = _block64(x, w, "1b", cos[ctx:], sin[ctx:], k[i], v[i], ctx)
    return {"logits": _norm64(x, t["norm"]) @ t["out"].double().t(), "k": k, "v": v}

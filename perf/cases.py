"""The work that a user of the framework has it do, as timed cases.

Each case is one pass through a public entry point: a normalisation, a rotary
embedding, a linear layer, a feed-forward block, an attention call, an
attention layer, or a whole model's prefill or decode step. `listed()` names
the cases, `draw(rng)` gives more of the same ranges, `prepare` makes what a
program holds before the call, `run` is the call, `exact` the same result in
64 bits from plain torch.
"""
from __future__ import annotations

import math

import torch

from torchplusplus_amd.attention import (GroupedQueryAttention, MultiHeadAttention,
                                         MultiQueryAttention, SlidingWindowAttention,
                                         decode_attention, flash_attn_func)
from torchplusplus_amd.dlops.linear import (LinearGELU, LinearNBBf16, LinearNBFp16, LinearRELU,
                                            LinearSILU)
from torchplusplus_amd.dlops.normalization import LayerNormFused, RmsNormFused
from torchplusplus_amd.dlops.rope import qkrope_apply
from torchplusplus_amd.fastqwen3 import FFN, FastQwen3, QwenConfig
from torchplusplus_amd.llmops.kvcache import KVCache

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-6
VOCAB, EMBED, LAYERS, HEADS, KV_HEADS, HEAD_DIM, HIDDEN = 151936, 1024, 28, 16, 8, 128, 3072
THETA = 1e6
# the costliest listed case is the feed-forward block over 16384 tokens; drawn
# cases stay below its operations and below this many attention scores
MAX_SCORES = 4 * 16 * 2048 * 2048
MAX_FLOPS = 2.9e11


def listed():
    return [
        # one decode token through a plain projection, the smallest call there is
        {"name": "gemv-1x1024x3072", "op": "linear", "act": "none", "bias": False, "rows": 1,
         "n_in": 1024, "n_out": 3072, "dtype": "fp16"},
        # a prompt's normalisation
        {"name": "rmsnorm-4096x1024", "op": "norm", "kind": "rms", "rows": 4096, "hidden": 1024,
         "dtype": "fp16"},
        # rotary embedding of a prompt's queries and keys
        {"name": "rope-qk-2048", "op": "rope", "batch": 1, "heads": 16, "kv_heads": 8,
         "seq": 2048, "head_dim": 128, "dtype": "bf16"},
        # a prompt of ordinary length through a fused linear layer
        {"name": "linear-silu-2048", "op": "linear", "act": "silu", "bias": True, "rows": 2048,
         "n_in": 1024, "n_out": 3072, "dtype": "bf16"},
        # a short prompt (or a batch of decode tokens) through a fused linear layer
        {"name": "linear-gelu-77", "op": "linear", "act": "gelu", "bias": True, "rows": 77,
         "n_in": 3072, "n_out": 1024, "dtype": "fp16"},
        # the feed-forward block over a batch of eight 2048-token prompts
        {"name": "ffn-16384", "op": "ffn", "rows": 16384, "n_in": 1024, "hidden": 3072,
         "dtype": "bf16"},
        # causal attention over a batch of prompts
        {"name": "attn-causal-4x2048", "op": "attn", "batch": 4, "heads": 16, "kv_heads": 8,
         "seq_q": 2048, "seq_k": 2048, "head_dim": 128, "causal": True, "window": -1,
         "dtype": "bf16"},
        # a follow-up turn: 200 new tokens against a conversation already cached
        {"name": "attn-append-200", "op": "attn", "batch": 1, "heads": 16, "kv_heads": 8,
         "seq_q": 200, "seq_k": 3001, "head_dim": 128, "causal": True, "window": -1,
         "dtype": "bf16"},
        # decode over a serving batch of 32 sequences of mixed lengths, in
        # caches with room for 8192 positions
        {"name": "decode-attn-32", "op": "decode", "batch": 32, "heads": 16, "kv_heads": 8,
         "min_len": 100, "max_len": 4096, "capacity": 8192, "head_dim": 128, "dtype": "bf16"},
        # a sliding-window attention layer over two ragged-length prompts
        {"name": "swa-layer-2x1000", "op": "layer", "kind": "swa", "batch": 2, "seq": 1000,
         "embed": 1024, "heads": 16, "head_dim": 64, "window": 512, "past": 0, "capacity": 0,
         "dtype": "bf16"},
        # the whole model on one short prompt
        {"name": "model-prefill-230", "op": "model", "batch": 1, "seq": 230, "past": 0,
         "capacity": 512, "dtype": "bf16"},
        # one decode step of the whole model for four sequences
        {"name": "model-decode-4", "op": "model", "batch": 4, "seq": 1, "past": 900,
         "capacity": 1280, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["linear", "linear", "linear", "norm", "rope", "ffn", "attn", "attn",
                     "decode", "decode", "layer", "layer", "model"])
    case = {"op": op, "dtype": rng.choice(["fp16", "bf16"])}
    if op == "linear":
        n_in, n_out = rng.choice([(1024, 3072), (3072, 1024), (1024, 4096), (2048, 1024),
                                  (1024, 1024), (768, 3072), (2048, 5632), (4096, 1000),
                                  (1000, 2048)])
        case.update(act=rng.choice(["none", "silu", "gelu", "relu"]), bias=rng.random() < 0.5,
                    rows=min(_log(rng, 1, 16384), int(MAX_FLOPS / (2 * n_in * n_out))),
                    n_in=n_in, n_out=n_out)
        if case["act"] == "none":
            case["bias"] = False
    elif op == "norm":
        hidden = rng.choice([128, 768, 1000, 1024, 1025, 2048, 4096, 8192])
        case.update(kind=rng.choice(["rms", "layer"]), hidden=hidden,
                    rows=_log(rng, 1, min(32768, (1 << 26) // hidden)))
    elif op == "rope":
        heads = rng.choice([8, 16, 32])
        case.update(batch=rng.choice([1, 2, 4]), heads=heads,
                    kv_heads=heads // rng.choice([1, 2, 4]), seq=_log(rng, 16, 8192),
                    head_dim=rng.choice([64, 128]))
    elif op == "ffn":
        n_in, hidden = rng.choice([(1024, 3072), (768, 2048), (2048, 5632)])
        case.update(rows=min(_log(rng, 1, 16384), int(MAX_FLOPS / (6 * n_in * hidden))),
                    n_in=n_in, hidden=hidden)
    elif op == "attn":
        heads = rng.choice([8, 16, 32])
        batch, seq_q = rng.choice([1, 1, 2, 4]), _log(rng, 17, 4096)
        past = rng.choice([0, 0, _log(rng, 16, 8192)])
        seq_q = min(seq_q, int(math.sqrt(MAX_SCORES / (batch * heads))))
        past = min(past, MAX_SCORES // (batch * heads * seq_q) - seq_q)
        causal = rng.random() < 0.75
        case.update(batch=batch, heads=heads, kv_heads=heads // rng.choice([1, 2, 4, 8]),
                    seq_q=seq_q, seq_k=seq_q + past, head_dim=rng.choice([64, 128]),
                    causal=causal, window=rng.choice([-1, -1, 255, 511]) if causal else -1)
    elif op == "decode":
        heads, group = rng.choice([8, 16, 32]), rng.choice([1, 2, 4, 8])
        capacity, batch = rng.choice([512, 2048, 4096, 8192, 16384]), _log(rng, 1, 64)
        batch = max(1, min(batch, (32 * 8 * 8192) // (capacity * (heads // group))))
        max_len = _log(rng, 64, capacity)
        case.update(batch=batch, heads=heads, kv_heads=heads // group,
                    min_len=rng.choice([max_len, _log(rng, 32, max_len)]), max_len=max_len,
                    capacity=capacity, head_dim=rng.choice([64, 128]))
    elif op == "layer":
        kind, head_dim = rng.choice(["gqa", "gqa", "mha", "mqa", "swa"]), rng.choice([64, 128])
        past = rng.choice([0, _log(rng, 16, 4096)]) if kind == "gqa" else 0
        step = past > 0 and rng.random() < 0.5
        seq = 1 if step else _log(rng, 17, 2048)
        batch = _log(rng, 1, 32) if step else rng.choice([1, 2, 4])
        capacity = -(-(past + seq) // 256) * 256 if kind == "gqa" else 0
        case.update(kind=kind, batch=batch, seq=seq, embed=1024, heads=1024 // head_dim,
                    head_dim=head_dim, window=rng.choice([128, 512]) if kind == "swa" else -1,
                    past=past, capacity=capacity)
    else:
        step = rng.random() < 0.5
        past = _log(rng, 32, 1200) if step else 0
        batch = rng.choice([1, 2, 3, 4])
        seq = 1 if step else _log(rng, 17, 240 // batch)
        case.update(batch=batch, seq=seq, past=past,
                    capacity=-(-(past + seq) // 256) * 256, dtype="bf16")
    return case


# ---- shared pieces -------------------------------------------------------------


class _Maker:
    """Random tensors of one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        x = torch.empty(shape, dtype=dtype, device=DEV)
        return x.normal_(mean, std, generator=self.gen)

    def ints(self, high, shape):
        return torch.randint(0, high, shape, generator=self.gen, device=DEV)

    def lengths(self, case):
        """The batch's lengths: evenly spread, in an order of the seed."""
        n = case["batch"]
        order = torch.randperm(n, generator=self.gen, device=DEV)
        return torch.tensor(_spread(case), dtype=torch.int32, device=DEV)[order]


def _spread(case):
    n, lo, hi = case["batch"], case["min_len"], case["max_len"]
    return [hi if n == 1 else lo + (hi - lo) * i // (n - 1) for i in range(n)]


def _tables(length, dim, dtype=torch.float16):
    """Rotary tables [length, dim], in half precision as the framework makes them."""
    inv = 1.0 / (THETA ** (torch.arange(0, dim, 2, device=DEV).float() / dim))
    ang = torch.arange(length, device=DEV).float()[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=1)
    return torch.cos(ang).to(dtype), torch.sin(ang).to(dtype)


def _rms(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rotate(x, cos, sin):
    """x [..., S, D] in 64 bits with tables [S, D]."""
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos.double() + turned * sin.double()


def _attend(q, k, v, causal, window):
    """q [B, Hq, Sq, D], k and v [B, Hkv, Sk, D] in 64 bits -> [B, Sq, Hq, D]."""
    b, hq, sq, d = q.shape
    hkv, sk = k.shape[1], k.shape[2]
    rel = (torch.arange(sk, device=q.device)[None, :]
           - torch.arange(sq, device=q.device)[:, None] - (sk - sq))
    keep = torch.ones(sq, sk, dtype=torch.bool, device=q.device)
    if causal:
        keep &= rel <= 0
    if window >= 0:
        keep &= rel >= -window
    out = torch.empty(b, sq, hq, d, dtype=torch.float64, device=q.device)
    for i in range(b):
        for h in range(hq):
            kh, vh = k[i, h * hkv // hq], v[i, h * hkv // hq]
            s = (q[i, h] @ kh.t().contiguous()) / math.sqrt(d)
            s = s.masked_fill_(~keep, -math.inf)
            out[i, :, h] = torch.softmax(s, dim=-1) @ vh
    return out


def _heads(x, n, d):
    """[B, S, n*d] -> [B, n, S, d]."""
    b, s, _ = x.shape
    return x.view(b, s, n, d).transpose(1, 2).contiguous()


def _visible(sq, sk, causal, window):
    """Scores that the mask keeps, of one head."""
    if not causal:
        return sq * sk
    total = 0
    for i in range(sq):
        last = i + sk - sq
        total += last + 1 - max(0, last - window if window >= 0 else 0)
    return total


def _rel(case, factor=1.0):
    """Relative error of a result in the case's type: the unit roundoff is
    2^-9 (bf16) or 2^-12 (fp16), and a result is rounded a few times."""
    return {"rel": factor * (1e-2 if case["dtype"] == "bf16" else 1.5e-3)}


# ---- one layer or one call each -----------------------------------------------------


class _Norm:
    @staticmethod
    def inputs(case, make, dt):
        return {"x": make.normal((case["rows"], case["hidden"]), dt),
                "w": make.normal((case["hidden"],), dt, 0.1, 1.0)}

    @staticmethod
    def build(case, t, dt):
        cls = RmsNormFused if case["kind"] == "rms" else LayerNormFused
        mod = cls(case["hidden"], eps=EPS, dtype=dt, device=DEV)
        mod.load_state_dict({"weight": t["w"]})
        return {"mod": mod, "x": t["x"]}

    @staticmethod
    def run(s):
        return s["mod"](s["x"])

    @staticmethod
    def exact(case, t):
        x = t["x"].double()
        if case["kind"] == "rms":
            return _rms(x, t["w"])
        x = x - x.mean(-1, keepdim=True)
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * t["w"].double()

    @staticmethod
    def work(case):
        n = case["rows"] * case["hidden"]
        return {"bytes": 2 * (2 * n + case["hidden"]), "flops": 4 * n}


class _Rope:
    @staticmethod
    def inputs(case, make, dt):
        b, s, d = case["batch"], case["seq"], case["head_dim"]
        cos, sin = _tables(s, d)
        return {"q": make.normal((b, case["heads"], s, d), dt),
                "k": make.normal((b, case["kv_heads"], s, d), dt), "cos": cos, "sin": sin}

    @staticmethod
    def build(case, t, dt):
        return t

    @staticmethod
    def run(s):
        return qkrope_apply(s["q"], s["k"], s["cos"], s["sin"])

    @staticmethod
    def exact(case, t):
        return tuple(_rotate(t[n].double(), t["cos"], t["sin"]) for n in ("q", "k"))

    @staticmethod
    def work(case):
        n = case["batch"] * (case["heads"] + case["kv_heads"]) * case["seq"] * case["head_dim"]
        return {"bytes": 4 * n + 4 * case["seq"] * case["head_dim"], "flops": 3 * n}


class _Linear:
    MODS = {"silu": LinearSILU, "gelu": LinearGELU, "relu": LinearRELU}
    ACTS = {"silu": torch.nn.functional.silu, "relu": torch.relu, "none": lambda x: x,
            "gelu": lambda x: torch.nn.functional.gelu(x, approximate="tanh")}

    @staticmethod
    def inputs(case, make, dt):
        t = {"x": make.normal((case["rows"], case["n_in"]), dt),
             "w": make.normal((case["n_out"], case["n_in"]), dt, 0.02)}
        if case["bias"]:
            t["b"] = make.normal((case["n_out"],), dt, 0.02)
        return t

    @staticmethod
    def build(case, t, dt):
        n_in, n_out = case["n_in"], case["n_out"]
        if case["act"] == "none":
            cls = LinearNBFp16 if dt == torch.float16 else LinearNBBf16
            mod = cls(n_in, n_out).to(DEV)
            mod.load_state_dict({"linear.weight": t["w"]})
        else:
            mod = _Linear.MODS[case["act"]](n_in, n_out, bias=case["bias"], dtype=dt, device=DEV)
            mod.load_state_dict({"weight": t["w"], **({"bias": t["b"]} if "b" in t else {})})
        return {"mod": mod, "x": t["x"]}

    @staticmethod
    def run(s):
        return s["mod"](s["x"])

    @staticmethod
    def exact(case, t):
        y = t["x"].double() @ t["w"].double().t()
        if "b" in t:
            y = y + t["b"].double()
        return _Linear.ACTS[case["act"]](y)

    @staticmethod
    def work(case):
        m, k, n = case["rows"], case["n_in"], case["n_out"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}


class _Ffn:
    @staticmethod
    def inputs(case, make, dt):
        e, h = case["n_in"], case["hidden"]
        return {"x": make.normal((1, case["rows"], e), dt), "gate": make.normal((h, e), dt, 0.02),
                "up": make.normal((h, e), dt, 0.02), "down": make.normal((e, h), dt, 0.02)}

    @staticmethod
    def build(case, t, dt):
        mod = FFN(case["n_in"], case["hidden"], dtype=dt, device=DEV)
        mod.load_state_dict({"fused_linear_layer1.weight": t["gate"],
                             "linear_layerP.weight": t["up"], "linear_layer2.weight": t["down"]})
        mod.refresh_fused_weights()
        return {"mod": mod, "x": t["x"]}

    @staticmethod
    def run(s):
        return s["mod"](s["x"])

    @staticmethod
    def exact(case, t):
        return _ffn(t["x"].double(), t["gate"], t["up"], t["down"])

    @staticmethod
    def work(case):
        m, e, h = case["rows"], case["n_in"], case["hidden"]
        return {"bytes": 2 * (2 * m * e + 3 * e * h), "flops": 6 * m * e * h}


def _ffn(x, gate, up, down):
    g = torch.nn.functional.silu(x @ gate.double().t()) * (x @ up.double().t())
    return g @ down.double().t()


class _Attn:
    """flash_attn_func on q [B, S, H, D] and key/value rows [B, H, S, D] seen
    as [B, S, H, D], the layout of a cache prefix."""

    @staticmethod
    def inputs(case, make, dt):
        b, d = case["batch"], case["head_dim"]
        kv = (b, case["kv_heads"], case["seq_k"], d)
        return {"q": make.normal((b, case["seq_q"], case["heads"], d), dt),
                "k": make.normal(kv, dt), "v": make.normal(kv, dt)}

    @staticmethod
    def build(case, t, dt):
        return {"q": t["q"], "k": t["k"].transpose(1, 2), "v": t["v"].transpose(1, 2),
                "causal": case["causal"], "window": (case["window"], -1)}

    @staticmethod
    def run(s):
        return flash_attn_func(s["q"], s["k"], s["v"], causal=s["causal"],
                               window_size=s["window"])

    @staticmethod
    def exact(case, t):
        return _attend(t["q"].double().transpose(1, 2).contiguous(), t["k"].double(),
                       t["v"].double(), case["causal"], case["window"])

    @staticmethod
    def work(case):
        b, d, hq, hk = case["batch"], case["head_dim"], case["heads"], case["kv_heads"]
        n = _visible(case["seq_q"], case["seq_k"], case["causal"], case["window"])
        return {"bytes": 4 * b * d * (case["seq_q"] * hq + case["seq_k"] * hk),
                "flops": 4 * b * hq * d * n}


class _Decode:
    @staticmethod
    def inputs(case, make, dt):
        b, d = case["batch"], case["head_dim"]
        kv = (b, case["kv_heads"], case["capacity"], d)
        return {"q": make.normal((b, 1, case["heads"], d), dt), "k": make.normal(kv, dt),
                "v": make.normal(kv, dt), "lens": make.lengths(case)}

    @staticmethod
    def build(case, t, dt):
        return t

    @staticmethod
    def run(s):
        return decode_attention(s["q"], s["k"], s["v"], s["lens"])

    @staticmethod
    def exact(case, t):
        q, out = t["q"].double().transpose(1, 2).contiguous(), []
        for i, n in enumerate(t["lens"].tolist()):
            out.append(_attend(q[i:i + 1], t["k"][i:i + 1, :, :n].double(),
                               t["v"][i:i + 1, :, :n].double(), False, -1))
        return torch.cat(out)

    @staticmethod
    def work(case):
        d, keys = case["head_dim"], sum(_spread(case))
        return {"bytes": 4 * d * (keys * case["kv_heads"] + case["batch"] * case["heads"]),
                "flops": 4 * d * keys * case["heads"]}


class _Layer:
    """An attention layer: projections, per-head norm, rotary embedding,
    attention and output projection. The grouped-query layer runs through a
    cache that holds `past` positions."""

    @staticmethod
    def kv_heads(case):
        n = case["heads"]
        return {"gqa": n // 2, "mha": n, "swa": n, "mqa": 1}[case["kind"]]

    @staticmethod
    def inputs(case, make, dt):
        e, d, hq, hk = case["embed"], case["head_dim"], case["heads"], _Layer.kv_heads(case)
        t = {"x": make.normal((case["batch"], case["seq"], e), dt)}
        for name, rows, cols in (("Wq", hq * d, e), ("Wk", hk * d, e), ("Wv", hk * d, e),
                                 ("out_projection", e, hq * d)):
            t[f"{name}.weight"] = make.normal((rows, cols), dt, 0.02)
        if case["kind"] in ("mha", "swa"):
            t["out_projection.bias"] = make.normal((e,), dt, 0.02)
        for name in ("q_norm", "k_norm"):
            t[f"{name}.weight"] = make.normal((d,), dt, 0.1, 1.0)
        if case["capacity"]:
            past = (case["batch"], hk, case["past"], d)
            t["k"], t["v"] = make.normal(past, dt), make.normal(past, dt, 0.64)
        t["cos"], t["sin"] = _tables(max(case["seq"], case["capacity"]), d)
        return t

    @staticmethod
    def build(case, t, dt):
        e, n, kind = case["embed"], case["heads"], case["kind"]
        if kind == "gqa":
            mod = GroupedQueryAttention(e, n, n // 2, case["head_dim"], dtype=dt, device=DEV)
        elif kind == "mha":
            mod = MultiHeadAttention(e, n, dtype=dt, device=DEV)
        elif kind == "mqa":
            mod = MultiQueryAttention(n, e, dtype=dt, device=DEV)
        else:
            mod = SlidingWindowAttention(case["window"], e, n, dtype=dt, device=DEV)
        mod.load_state_dict({k: v for k, v in t.items() if "." in k})
        s = {"mod": mod, "x": t["x"], "cos": t["cos"], "sin": t["sin"], "cache": None,
             "past": case["past"]}
        if kind == "gqa":
            mod.refresh_fused_weights()
            cache = KVCache(case["capacity"], n // 2, case["head_dim"], dt, DEV, case["batch"])
            if case["past"]:
                cache.update(t["k"], t["v"])
            s["cache"] = cache
        return s

    @staticmethod
    def run(s):
        with torch.inference_mode():
            if s["cache"] is None:
                return s["mod"](s["x"], s["cos"], s["sin"])
            out = s["mod"](s["x"], s["cos"], s["sin"], s["cache"], s["past"])
            return out, s["cache"].k_cache, s["cache"].v_cache

    @staticmethod
    def exact(case, t):
        d, hq, hk, past = case["head_dim"], case["heads"], _Layer.kv_heads(case), case["past"]
        x = t["x"].double()
        w = {n: t[f"{n}.weight"].double().t() for n in ("Wq", "Wk", "Wv", "out_projection")}
        q, k, v = (_heads(x @ w[n], c, d) for n, c in (("Wq", hq), ("Wk", hk), ("Wv", hk)))
        q, k = _rms(q, t["q_norm.weight"]), _rms(k, t["k_norm.weight"])
        rows = slice(past, past + case["seq"])
        q, k = (_rotate(y, t["cos"][rows], t["sin"][rows]) for y in (q, k))
        if case["capacity"]:
            k, v = torch.cat([t["k"].double(), k], 2), torch.cat([t["v"].double(), v], 2)
        window = case["window"] - 1 if case["kind"] == "swa" else -1
        o = _attend(q, k, v, True, window).reshape(*x.shape[:2], hq * d) @ w["out_projection"]
        if "out_projection.bias" in t:
            o = o + t["out_projection.bias"].double()
        if not case["capacity"]:
            return o
        pad = (0, 0, 0, case["capacity"] - past - case["seq"])
        return o, torch.nn.functional.pad(k, pad), torch.nn.functional.pad(v, pad)

    @staticmethod
    def work(case):
        e, d, hq, hk = case["embed"], case["head_dim"], case["heads"], _Layer.kv_heads(case)
        m, total = case["batch"] * case["seq"], case["past"] + case["seq"]
        weights = e * d * (2 * hq + 2 * hk)
        window = case["window"] - 1 if case["kind"] == "swa" else -1
        n = _visible(case["seq"], total, True, window)
        kept = 2 * case["batch"] * hk * d * total if case["capacity"] else 0
        return {"bytes": 2 * (2 * m * e + weights + kept),
                "flops": 2 * m * weights + 4 * case["batch"] * hq * d * n}


class _Model:
    """The Qwen3-0.6B-shape decoder: a prompt's prefill (the last position's
    logits, as generation uses them) or one decode step, through caches that
    already hold `past` positions."""

    @staticmethod
    def inputs(case, make, dt):
        t = {"tok_embed.weight": make.normal((VOCAB, EMBED), dt, 0.02),
             "out_head.weight": make.normal((VOCAB, EMBED), dt, 0.02),
             "final_rmsnorm.weight": make.normal((EMBED,), dt, 0.1, 1.0)}
        q, kv = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
        for i in range(LAYERS):
            p = f"transformer_blocs.{i}."
            for name, rows, cols in (
                    ("attn.Wq", q, EMBED), ("attn.Wk", kv, EMBED), ("attn.Wv", kv, EMBED),
                    ("attn.out_projection", EMBED, q), ("ffn.fused_linear_layer1", HIDDEN, EMBED),
                    ("ffn.linear_layerP", HIDDEN, EMBED), ("ffn.linear_layer2", EMBED, HIDDEN)):
                t[f"{p}{name}.weight"] = make.normal((rows, cols), dt, 0.02)
            for name, n in (("attn.q_norm", HEAD_DIM), ("attn.k_norm", HEAD_DIM),
                            ("rms_norm1", EMBED), ("rms_norm2", EMBED)):
                t[f"{p}{name}.weight"] = make.normal((n,), dt, 0.1, 1.0)
        t["ids"] = make.ints(VOCAB, (case["batch"], case["seq"]))
        if case["past"]:
            past = (LAYERS, case["batch"], KV_HEADS, case["past"], HEAD_DIM)
            t["k"], t["v"] = make.normal(past, dt), make.normal(past, dt, 0.64)
        return t

    @staticmethod
    def build(case, t, dt):
        model = FastQwen3(QwenConfig(dtype=dt), device=DEV, rope_context=4096)
        model.load_state_dict({k: v for k, v in t.items() if k.endswith(".weight")})
        model.refresh_fused_weights()
        model.setup_kv_cache(case["capacity"], case["batch"])
        if case["past"]:
            for i, cache in enumerate(model.kv_cache_array):
                cache.update(t["k"][i], t["v"][i])
        return {"model": model, "ids": t["ids"], "past": case["past"]}

    @staticmethod
    def run(s):
        model = s["model"]
        with torch.inference_mode():
            logits = model.forward_impl(s["ids"], model.kv_cache_array, s["past"], last_only=True)
        return (logits, [c.k_cache for c in model.kv_cache_array],
                [c.v_cache for c in model.kv_cache_array])

    @staticmethod
    def exact(case, t):
        past, rows = case["past"], slice(case["past"], case["past"] + case["seq"])
        cos, sin = _tables(4096, HEAD_DIM)
        pad = (0, 0, 0, case["capacity"] - past - case["seq"])
        x, ks, vs = t["tok_embed.weight"][t["ids"]].double(), [], []
        for i in range(LAYERS):
            w = {n[len(f"transformer_blocs.{i}."):-len(".weight")]: v for n, v in t.items()
                 if n.startswith(f"transformer_blocs.{i}.")}
            h = _rms(x, w["rms_norm1"])
            q, k, v = (_heads(h @ w[f"attn.W{n}"].double().t(), c, HEAD_DIM)
                       for n, c in (("q", HEADS), ("k", KV_HEADS), ("v", KV_HEADS)))
            q = _rotate(_rms(q, w["attn.q_norm"]), cos[rows], sin[rows])
            k = _rotate(_rms(k, w["attn.k_norm"]), cos[rows], sin[rows])
            if past:
                k = torch.cat([t["k"][i].double(), k], 2)
                v = torch.cat([t["v"][i].double(), v], 2)
            o = _attend(q, k, v, True, -1).reshape(*x.shape[:2], HEADS * HEAD_DIM)
            x = x + o @ w["attn.out_projection"].double().t()
            x = x + _ffn(_rms(x, w["rms_norm2"]), w["ffn.fused_linear_layer1"],
                         w["ffn.linear_layerP"], w["ffn.linear_layer2"])
            ks.append(torch.nn.functional.pad(k, pad))
            vs.append(torch.nn.functional.pad(v, pad))
        x = _rms(x[:, -1:], t["final_rmsnorm.weight"])
        return x @ t["out_head.weight"].double().t(), ks, vs

    @staticmethod
    def work(case):
        m, total = case["batch"] * case["seq"], case["past"] + case["seq"]
        layer = EMBED * (2 * HEADS * HEAD_DIM + 2 * KV_HEADS * HEAD_DIM + 3 * HIDDEN)
        n = _visible(case["seq"], total, True, -1)
        cached = 2 * case["batch"] * KV_HEADS * HEAD_DIM * total
        return {"bytes": 2 * (LAYERS * (layer + cached) + VOCAB * EMBED + m * EMBED
                              + case["batch"] * VOCAB),
                "flops": LAYERS * (2 * m * layer + 4 * case["batch"] * HEADS * HEAD_DIM * n)
                + 2 * case["batch"] * VOCAB * EMBED}


_OPS = {"norm": _Norm, "rope": _Rope, "linear": _Linear, "ffn": _Ffn, "attn": _Attn,
        "decode": _Decode, "layer": _Layer, "model": _Model}


def prepare(case, seed):
    op, dt = _OPS[case["op"]], DTYPES[case["dtype"]]
    return op, op.build(case, op.inputs(case, _Maker(seed), dt), dt)


def run(state):
    op, s = state
    return op.run(s)


def work(case):
    return _OPS[case["op"]].work(case)


def tolerance(case):
    # A layer rounds at every operation between its projections. A whole model
    # carries the roundings of 28 of them: the same decode step through the
    # 4-row and the 20-row kernels differs by 3e-2 (random caches, over which
    # attention averages nearly uniformly), a prompt by about a third of that.
    if case["op"] == "model":
        return _rel(case, 12.0 if case["past"] else 5.0)
    return _rel(case, 1.5 if case["op"] == "layer" else 1.0)


def exact(case, seed):
    op, dt = _OPS[case["op"]], DTYPES[case["dtype"]]
    with torch.no_grad():
        return op.exact(case, op.inputs(case, _Maker(seed), dt))

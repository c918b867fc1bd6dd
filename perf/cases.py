"""Performance cases of the framework: single requests, batches, long shared prefixes and greedy decode
over the synthetic models of the workload shapes, through the Python binding of the C ABI.

Each case runs one call of a user's program on a model that the program keeps loaded; a model is cut to a
few of its equal layers where a whole one would add only repeats (`layers`).  `exact` restates every family
in float64 with torch, from the bytes of the model file.
"""
import functools
import json
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "laya-goish_amd"))

import laya_hip as lh  # noqa: E402

MODEL_SEED = 20261201
PRECISION = {"exact": lh.PREC_EXACT, "kv16": lh.PREC_KV16, "fast": lh.PREC_FAST}

# The dimensions that work() counts with; `mat` gives the file bytes of a weight: q|k, v, o, gate|up, down, head.
F16B, Q8B, Q4B, Q6B = 2.0, 34 / 32, 144 / 256, 210 / 256
SHAPES = {
    "plumbing-f16": dict(d=512, hq=8, hkv=8, hd=64, f=1408, V=32000, ctx=2048, mat=(F16B,) * 6),
    "q8-2048": dict(d=2048, hq=16, hkv=16, hd=128, f=5632, V=32000, ctx=4096, mat=(Q8B,) * 6),
    "q4km-7b": dict(d=3584, hq=28, hkv=4, hd=128, f=18944, V=152064, ctx=4096, mat=(Q4B, Q6B, Q4B, Q4B, Q6B, Q6B)),
    "f16-7b": dict(d=3584, hq=28, hkv=4, hd=128, f=18944, V=152064, ctx=10240, mat=(F16B,) * 6),
    "openthai-0.8b": dict(d=1024, f=3584, V=248339, ctx=4096),
    "laya-english": dict(d=768, f=1152, V=50368, ctx=512, head_f=768),
}
# Layers that a drawn case of each model runs.
DRAWN_LAYERS = {"plumbing-f16": 6, "q8-2048": 4, "q4km-7b": 2, "f16-7b": 2, "openthai-0.8b": 4, "laya-english": 6}


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest call: one yes/no decision of the small F16 model, a whole model; launches and latency count
        dict(name="plumbing_request", call="batch", model="plumbing-f16", layers=6, precision="exact", requests=1,
             shortest=144, longest=144, prefix=0, positions=1),
        # a short classification with the encoder, the whole model
        dict(name="laya_request", call="encode", model="laya-english", layers=22, precision="exact", requests=1,
             shortest=45, longest=45, options=2),
        # a server's full batch of encoder inputs near the context length, lengths ragged
        dict(name="laya_batch", call="encode", model="laya-english", layers=6, precision="exact", requests=64,
             shortest=473, longest=512, options=4),
        # one long choice over many options: linear-attention layers and a full-attention layer at an odd length
        dict(name="openthai_request", call="batch", model="openthai-0.8b", layers=4, precision="exact", requests=1,
             shortest=1437, longest=1437, prefix=0, positions=1),
        # one short question in eight option orders, all as one batch
        dict(name="openthai_passes", call="batch", model="openthai-0.8b", layers=4, precision="exact", requests=8,
             shortest=57, longest=63, prefix=0, positions=1),
        # one decision on the 8-bit model: a few hundred tokens, three questions
        dict(name="q8_request", call="batch", model="q8-2048", layers=4, precision="exact", requests=1, shortest=301,
             longest=301, prefix=0, positions=3),
        # the headline workload: 64 independent requests with three questions each
        dict(name="q8_batch", call="batch", model="q8-2048", layers=4, precision="exact", requests=64, shortest=521,
             longest=560, prefix=0, positions=3),
        # greedy text after a long context, batch 1: bound by weight and cache bytes
        dict(name="q8_decode", call="decode", model="q8-2048", layers=4, precision="exact", context=2048, steps=16),
        # the same on the mixed 4/6-bit 7B shape with grouped heads
        dict(name="q4k_decode", call="decode", model="q4km-7b", layers=2, precision="exact", context=1021, steps=16),
        # one decision on the 7B shape with the half-size cache
        dict(name="q4k_request_kv16", call="batch", model="q4km-7b", layers=2, precision="kv16", requests=1,
             shortest=700, longest=700, prefix=0, positions=3),
        # batched prefill of the 4/6-bit 7B shape
        dict(name="q4k_batch", call="batch", model="q4km-7b", layers=2, precision="exact", requests=16, shortest=1000,
             longest=1024, prefix=0, positions=1),
        # long context: requests that go on from a cached common prefix, F16 7B shape
        dict(name="f16_prefix", call="batch", model="f16-7b", layers=2, precision="exact", requests=8, shortest=2048,
             longest=2048, prefix=6144, positions=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["one", "one", "batch", "encode", "decode", "prefix"])
    if call == "encode":
        longest = _log_int(rng, 17, 512)
        requests = max(1, min(_log_int(rng, 1, 64), 16384 // longest))
        return dict(call="encode", model="laya-english", layers=6, precision="exact", requests=requests,
                    shortest=max(17, longest - rng.randint(0, longest // 4)), longest=longest,
                    options=rng.randint(2, 16))
    if call == "decode":
        model = rng.choice(["q8-2048", "q4km-7b", "f16-7b", "plumbing-f16"])
        return dict(call="decode", model=model, layers=DRAWN_LAYERS[model], precision=rng.choice(["exact", "exact", "kv16"]),
                    context=_log_int(rng, 16, SHAPES[model]["ctx"] // 2 - 64), steps=rng.randint(2, 24))
    if call == "prefix":
        model = rng.choice(["q8-2048", "q4km-7b", "f16-7b"])
        longest, prefix = _log_int(rng, 32, 1024), _log_int(rng, 64, 3000)
        requests, shortest = rng.randint(1, 8), longest - rng.randint(0, longest // 3)
        return dict(call="batch", model=model, layers=DRAWN_LAYERS[model], precision=rng.choice(["exact", "exact", "kv16"]),
                    requests=requests, shortest=shortest, longest=longest, prefix=prefix, positions=rng.randint(1, 4))
    model = rng.choice(["plumbing-f16", "q8-2048", "q4km-7b", "f16-7b", "openthai-0.8b"])
    precision = rng.choice({"openthai-0.8b": ["exact"], "plumbing-f16": ["exact", "fast"]}.get(model, ["exact", "exact", "kv16"]))
    longest = _log_int(rng, 24, 1500)
    requests = 1 if call == "one" else max(2, min(_log_int(rng, 2, 48), 12288 // longest))
    shortest = longest if requests == 1 else longest - rng.randint(0, longest // 3)
    return dict(call="batch", model=model, layers=DRAWN_LAYERS[model], precision=precision, requests=requests,
                shortest=shortest, longest=longest, prefix=0, positions=rng.randint(1, 4))


def _lengths(case):
    """Tokens of each request: spread over [shortest, longest], neighbours unlike."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    return [hi] if n == 1 else [lo + (hi - lo) * (i * 29 % n) // (n - 1) for i in range(n)]


def _positions(n, count):
    """`count` answer positions of a request of n tokens, the last token's among them."""
    return sorted({n - 1 - i * (n // (count + 1)) for i in range(count)})


# ------------------------------------------------------------------ a user's program
@functools.lru_cache(maxsize=None)
def _engine(model, layers, precision):
    """The loaded model, kept for the life of the program as a server keeps it."""
    gguf = lh.Gguf.from_bytes(lh.SynthImage(model, MODEL_SEED, layers))
    return lh.Engine(gguf, kv_tokens=131072, precision=PRECISION[precision])


class _State:
    """The request data of a case and the sequences that the program holds between calls."""

    def __init__(self, case, engine, inputs):
        self.case, self.engine, self.inputs, self.held = case, engine, inputs, []

    def __del__(self):
        for s in self.held:
            self.engine.seq_free(s)


def _inputs(case, seed):
    rng, s = np.random.RandomState(seed % (1 << 32)), SHAPES[case["model"]]
    draw_ids = lambda n: rng.randint(0, s["V"], n).astype(np.int32)  # noqa: E731
    if case["call"] == "encode":
        return [(draw_ids(n), np.sort(rng.choice(n, case["options"], replace=False)).astype(np.int32), int(rng.randint(3)))
                for n in _lengths(case)]
    if case["call"] == "decode":
        return {"context": draw_ids(case["context"]), "first": int(draw_ids(1)[0])}
    return {"prefix": draw_ids(case["prefix"]),
            "requests": [(draw_ids(n), np.array(_positions(n, case["positions"]), np.int32)) for n in _lengths(case)]}


def _option_rows(model):
    """Head rows that a decision reads: the 256 option slots (the top of a decoder's vocabulary)."""
    v = 256 if model == "openthai-0.8b" else SHAPES[model]["V"]
    return np.arange(v - 256, v, dtype=np.int32)


def prepare(case, seed):
    engine = _engine(case["model"], case["layers"], case["precision"])
    state = _State(case, engine, _inputs(case, seed))
    before = state.inputs["context" if case["call"] == "decode" else "prefix"] if case["call"] != "encode" else ()
    if len(before):  # tokens that are in the cache before the call
        seq = engine.seq_create()
        state.held.append(seq)
        engine.forward(seq, before, [len(before) - 1], vocab_ids=[0])
    return state


def run(state):
    case, engine, inputs = state.case, state.engine, state.inputs
    if case["call"] == "encode":
        out = engine.laya_forward(inputs)
        return {"logits": np.stack([logits for logits, _ in out]), "act": np.stack([act for _, act in out])}
    if case["call"] == "decode":  # a greedy run, then the distribution after it
        seq = engine.seq_fork(state.held[0], case["context"])
        try:
            tokens = engine.decode(seq, inputs["first"], case["steps"] - 1)
            _, logits = engine.decode(seq, int(tokens[-1]), 1, want_logits=True)
        finally:
            engine.seq_free(seq)
        return {"tokens": tokens, "logits": logits[0]}
    seqs = [engine.seq_fork(state.held[0], case["prefix"]) if case["prefix"] else engine.seq_create()
            for _ in inputs["requests"]]
    try:
        batch = engine.batch([(s, ids, pos) for s, (ids, pos) in zip(seqs, inputs["requests"])])
        logits = batch.run(_option_rows(case["model"]))[0]
        batch.free()
    finally:
        for s in seqs:
            engine.seq_free(s)
    return {"logits": logits}


# ------------------------------------------------------------------ the work of a call
def _decoder_layer(s):
    """(weights, file bytes) of a decoder layer's matrices."""
    d, q, kv, f, m = s["d"], s["hq"] * s["hd"], s["hkv"] * s["hd"], s["f"], s["mat"]
    parts = [(d * (q + kv), m[0]), (d * kv, m[1]), (q * d, m[2]), (d * 2 * f, m[3]), (f * d, m[4])]
    return sum(n for n, _ in parts), sum(n * b for n, b in parts)


def work(case):
    s, layers = SHAPES[case["model"]], case["layers"]
    d, f = s["d"], s["f"]
    if case["call"] == "decode":
        weights, size = _decoder_layer(s)
        keys = sum(case["context"] + i + 1 for i in range(case["steps"]))
        kv_bytes = (4 if case["precision"] == "exact" else 2) * 2 * s["hkv"] * s["hd"]
        return {"bytes": case["steps"] * (layers * size + s["V"] * d * s["mat"][5]) + layers * keys * kv_bytes + 4 * s["V"],
                "flops": case["steps"] * 2 * (layers * weights + s["V"] * d) + layers * keys * 4 * s["hq"] * s["hd"]}
    lengths = _lengths(case)
    tokens = sum(lengths)
    if case["call"] == "encode":
        every = layers * (4 * d * d + 3 * d * f) + 2 * (4 * d * d + 2 * d * s["head_f"])
        full = (layers + 2) // 3 + 2
        pairs = sum(n * n * full + (layers + 2 - full) * sum(min(n, i + 65) - max(0, i - 64) for i in range(n)) for n in lengths)
        return {"bytes": 2 * every + 2 * tokens * d + 4 * len(lengths) * (case["options"] + 2),
                "flops": 2 * every * tokens + 4 * d * pairs}
    rows = sum(len(_positions(n, case["positions"])) for n in lengths)
    pairs = sum(n * case["prefix"] + n * (n + 1) // 2 for n in lengths)
    if case["model"] == "openthai-0.8b":
        full = layers // 4
        mixer = (layers - full) * (d * (4 * 2048 + 32) + 2048 * d) + full * (d * (4096 + 1024) + 2048 * d)
        every = mixer + layers * 3 * d * f
        return {"bytes": 2 * every + 2 * tokens * d + 2 * 256 * d + 4 * rows * 256,
                "flops": 2 * every * tokens + full * pairs * 4 * 2048 + (layers - full) * tokens * 16 * 128 * 128 * 7 + 2 * rows * 256 * d}
    weights, size = _decoder_layer(s)
    kv_bytes = layers * (4 if case["precision"] == "exact" else 2) * 2 * s["hkv"] * s["hd"]
    return {"bytes": layers * size + 2 * tokens * d + kv_bytes * (case["prefix"] + tokens) + 256 * d * s["mat"][5] + 4 * rows * 256,
            "flops": 2 * layers * weights * tokens + layers * pairs * 4 * s["hq"] * s["hd"] + 2 * rows * 256 * d}


# Four times the 2-norm distance to float64 that the call shows over these ranges.  Split f16 planes carry about 22 bits,
# so the exact mode differs by f32 summation orders, the 8- and 4-bit models' weights multiplying them; a cache or a
# weight in 16 bits brings its own rounding.  The encoder's few logits spread by sample: its bound is the worst one's.
REL = {("plumbing-f16", "exact"): 4e-6, ("plumbing-f16", "kv16"): 1.2e-3, ("plumbing-f16", "fast"): 2.8e-3,
       ("q8-2048", "exact"): 1e-4, ("q8-2048", "kv16"): 4e-2, ("q4km-7b", "exact"): 8e-5, ("q4km-7b", "kv16"): 2.5e-2,
       ("f16-7b", "exact"): 1.3e-5, ("f16-7b", "kv16"): 2.4e-3, ("openthai-0.8b", "exact"): 1.3e-5,
       ("laya-english", "exact"): 4e-5}


def tolerance(case):
    return {"rel": REL[case["model"], case["precision"]]}


# ------------------------------------------------------------------ float64
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _values(kind, raw):
    """Weights in float64 from the bytes of GGUF blocks (a flat uint8 tensor)."""
    if kind == lh.F32:
        return raw.view(torch.float32).double()
    if kind == lh.F16:
        return raw.view(torch.float16).double()
    if kind == lh.Q8_0:
        c = raw.view(-1, 34)
        return (_half(c[:, :2]) * c[:, 2:].contiguous().view(torch.int8).double()).flatten()
    if kind == lh.Q4_K:
        c = raw.view(-1, 144)
        s = c[:, 4:16].int()
        scale = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double() * _half(c[:, :2])
        low = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double() * _half(c[:, 2:4])
        n = c[:, 16:].view(-1, 4, 1, 32)
        codes = torch.cat([n & 15, n >> 4], 2).view(-1, 8, 32).double()
        return (codes * scale[:, :, None] - low[:, :, None]).flatten()
    if kind == lh.Q6_K:
        c = raw.view(-1, 210)
        ql, qh = c[:, :128].view(-1, 2, 2, 32), c[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)                                   # [block][half][4][32]
        high = torch.cat([(qh >> 2 * j) & 3 for j in range(4)], 2)
        codes = (low.int() + (high.int() << 4) - 32).double().view(-1, 16, 16)
        scale = c[:, 192:208].contiguous().view(torch.int8).double() * _half(c[:, 208:])
        return (codes * scale[:, :, None]).flatten()
    raise ValueError(kind)


class _File:
    """Tensors of a model file as float64."""

    def __init__(self, gguf):
        self.gguf, self.known = gguf, set(gguf.names())

    def __contains__(self, name):
        return name in self.known

    def rows(self, name, rows=None):
        kind, dims, raw = self.gguf.tensor(name)
        raw = torch.from_numpy(np.frombuffer(bytearray(raw), np.uint8))
        if rows is not None:
            raw = raw.view(int(np.prod(dims[1:])), -1)[torch.as_tensor(rows, dtype=torch.long)].flatten()
        v = _values(kind, raw.to(_device()))
        return v.view(-1, dims[0]) if len(dims) > 1 else v

    __call__ = rows


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rotate(x, cos, sin, half):
    """Pairs (j, j + half) of the first 2 * half dims of x [tokens][heads][dim] turned by tables [tokens][half]."""
    u, v, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
    c, s = cos[:, None, :half], sin[:, None, :half]
    return torch.cat([u * c - v * s, v * c + u * s, rest], -1)


def _attend(q, k, v, allowed):
    """q [n][heads][dim], k and v [m][kv heads][dim], allowed [n][m] or None, one head after another."""
    group = q.shape[1] // k.shape[1]
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // group].t().contiguous() / math.sqrt(q.shape[2])
        if allowed is not None:
            s = s.masked_fill(~allowed, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // group].contiguous()
    return out.flatten(1)


def _segments(lengths):
    at = np.cumsum([0] + list(lengths))
    return [slice(int(a), int(b)) for a, b in zip(at[:-1], at[1:])]


class _Decoder:
    def __init__(self, gguf, case):
        self.t, s = _File(gguf), SHAPES[case["model"]]
        self.hq, self.hkv, self.hd, self.f, self.layers = s["hq"], s["hkv"], s["hd"], s["f"], case["layers"]
        self.eps = float(np.float32(gguf.num("laya.decoder.layer_norm_rms_epsilon")))
        self.cos, self.sin = self.t("cos_full"), self.t("sin_full")
        self.w = [self._layer(str(i)) for i in range(self.layers)]
        self.final = self.t("final_norm.weight")

    def _layer(self, i):
        t = self.t
        parts = [f"qkv.{i}"] if f"qkv.{i}.weight" in t else [f"{p}.{i}" for p in "qkv"]
        bias = torch.cat([t(p + ".bias") for p in parts]) if parts[0] + ".bias" in t else 0.0
        return dict(qkv=torch.cat([t(p + ".weight") for p in parts]), bias=bias, wo=t(f"wo.{i}.weight"), wi=t(f"mlp_wi.{i}.weight"),
                    wd=t(f"mlp_wo.{i}.weight"), norm1=t(f"attn_norm.{i}.weight"), norm2=t(f"ffn_norm.{i}.weight"))

    def hidden(self, ids, caches):
        """Hidden states of the new tokens ids[r] behind caches[r] (a list of (k, v) of each layer, or empty), and the new caches."""
        lengths, starts = [len(i) for i in ids], [c[0][0].shape[0] if c else 0 for c in caches]
        segments, new = _segments(lengths), [[] for _ in ids]
        x = self.t("tok_emb.weight", np.concatenate(ids))
        pos = torch.cat([torch.arange(a, a + n) for a, n in zip(starts, lengths)]).to(x.device)
        cos, sin, qw, kw = self.cos[pos], self.sin[pos], self.hq * self.hd, self.hkv * self.hd
        for l, w in enumerate(self.w):
            qkv = _rms(x, w["norm1"], self.eps) @ w["qkv"].t() + w["bias"]
            q = _rotate(qkv[:, :qw].view(-1, self.hq, self.hd), cos, sin, self.hd // 2)
            k = _rotate(qkv[:, qw:qw + kw].view(-1, self.hkv, self.hd), cos, sin, self.hd // 2)
            v = qkv[:, qw + kw:].view(-1, self.hkv, self.hd)
            out = torch.empty(len(x), qw, dtype=x.dtype, device=x.device)
            for r, at in enumerate(segments):
                kr, vr = (torch.cat([caches[r][l][j], a[at]]) if caches[r] else a[at] for j, a in enumerate((k, v)))
                new[r].append((kr, vr))
                keys = torch.arange(kr.shape[0], device=x.device)
                out[at] = _attend(q[at], kr, vr, keys[None, :] <= pos[at][:, None])
            x = x + out @ w["wo"].t()
            g = _rms(x, w["norm2"], self.eps) @ w["wi"].t()
            x = x + (torch.nn.functional.silu(g[:, :self.f]) * g[:, self.f:]) @ w["wd"].t()
        return x, new

    def logits(self, x, head):
        return _rms(x, self.final, self.eps) @ head.t()


def _exact_decoder(case, inputs, gguf):
    m = _Decoder(gguf, case)
    if case["call"] == "decode":
        _, cache = m.hidden([inputs["context"]], [[]])
        head, token, tokens = m.t("output.weight"), inputs["first"], []
        for _ in range(case["steps"]):
            x, cache = m.hidden([np.array([token])], cache)
            logits = m.logits(x, head)[0]
            token = int(logits.argmax())
            tokens.append(token)
        return {"tokens": np.array(tokens[:-1], np.int32), "logits": logits.cpu().numpy()}
    cache = m.hidden([inputs["prefix"]], [[]])[1][0] if case["prefix"] else []
    ids, lengths = [i for i, _ in inputs["requests"]], _lengths(case)
    x, _ = m.hidden(ids, [cache] * len(ids))
    rows = np.concatenate([at.start + pos for at, (_, pos) in zip(_segments(lengths), inputs["requests"])])
    return {"logits": m.logits(x[torch.as_tensor(rows, device=x.device)], m.t("output.weight", _option_rows(case["model"]))).cpu().numpy()}


def _delta_rule(q, k, v, decay, beta):
    """Gated delta rule over tokens, q, k, v [requests][tokens][heads][128]: S <- a S + k (b (v - S^T k))^T, o = S^T q."""
    r, n, heads, w = q.shape
    state, out = torch.zeros(r, heads, w, w, dtype=q.dtype, device=q.device), torch.empty_like(v)
    for t in range(n):
        state = state * decay[:, t, :, None, None]
        kt = k[:, t, :, :, None]
        state = state + kt * (beta[:, t, :, None] * (v[:, t] - (state * kt).sum(2)))[:, :, None, :]
        out[:, t] = (state * q[:, t, :, :, None]).sum(2)
    return out


def _exact_openthai(case, inputs, gguf):
    t, cfg = _File(gguf), json.loads(gguf.str("openthai.config"))["text_config"]
    hq, hkv, nh, n_layers = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["linear_num_value_heads"], case["layers"]
    ids, lengths = [i for i, _ in inputs["requests"]], _lengths(case)
    segments, longest, wide = _segments(lengths), max(lengths), nh * 128
    x = t("model.embed_tokens.weight", np.concatenate(ids))
    # angles as the model defines them: position / theta^(2j/64) in 32 bits
    theta = (np.arange(longest, dtype=np.float32)[:, None] / np.float32(1e7) ** (np.arange(32, dtype=np.float32) * 2 / 64)).astype(np.float64)
    cos, sin = (torch.from_numpy(a).to(x.device) for a in (np.cos(theta), np.sin(theta)))
    norm = lambda x, name: _rms(x, 1.0 + t(name), 1e-6)  # noqa: E731

    def full(p, h):
        qg = (h @ t(p + "q_proj.weight").t()).view(-1, hq, 2, 256)
        k, v = ((h @ t(p + a + "_proj.weight").t()).view(-1, hkv, 256) for a in "kv")
        q, k, out = norm(qg[:, :, 0], p + "q_norm.weight"), norm(k, p + "k_norm.weight"), []
        for at, n in zip(segments, lengths):
            causal = torch.ones(n, n, dtype=torch.bool, device=h.device).tril()
            out.append(_attend(_rotate(q[at], cos[:n], sin[:n], 32), _rotate(k[at], cos[:n], sin[:n], 32), v[at], causal))
        return (torch.cat(out) * torch.sigmoid(qg[:, :, 1]).flatten(1)) @ t(p + "o_proj.weight").t()

    def delta(p, h):
        def padded(a):  # [requests][longest][...]: what follows a request's end does not reach its outputs
            out = torch.zeros(len(lengths), longest, *a.shape[1:], dtype=a.dtype, device=a.device)
            for r, (at, n) in enumerate(zip(segments, lengths)):
                out[r, :n] = a[at]
            return out

        raw, z, a, b = (h @ t(p + f"in_proj_{part}.weight").t() for part in ("qkv", "z", "a", "b"))
        taps, raw = t(p + "conv1d.weight").view(3 * wide, 4), torch.nn.functional.pad(padded(raw), (0, 0, 3, 0))
        qkv = torch.nn.functional.silu(sum(raw[:, j:j + longest] * taps[:, j] for j in range(4)))
        q, k, v = (c.reshape(len(lengths), longest, nh, 128) for c in qkv.split(wide, -1))
        unit = lambda a: a * torch.rsqrt((a * a).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        decay = torch.exp(-torch.exp(t(p + "A_log")) * torch.nn.functional.softplus(a + t(p + "dt_bias")))
        o = _delta_rule(unit(q) / math.sqrt(128), unit(k), v, padded(decay), padded(torch.sigmoid(b)))
        o = torch.cat([o[r, :n] for r, n in enumerate(lengths)])
        o = _rms(o, t(p + "norm.weight"), 1e-6).flatten(1) * torch.nn.functional.silu(z)
        return o @ t(p + "out_proj.weight").t()

    for l in range(n_layers):
        p = f"model.layers.{l}."
        h = norm(x, p + "input_layernorm.weight")
        x = x + (full(p + "self_attn.", h) if cfg["layer_types"][l] == "full_attention" else delta(p + "linear_attn.", h))
        h = norm(x, p + "post_attention_layernorm.weight")
        h = torch.nn.functional.silu(h @ t(p + "mlp.gate_proj.weight").t()) * (h @ t(p + "mlp.up_proj.weight").t())
        x = x + h @ t(p + "mlp.down_proj.weight").t()
    rows = np.concatenate([at.start + pos for at, (_, pos) in zip(segments, inputs["requests"])])
    x = norm(x[torch.as_tensor(rows, device=x.device)], "model.norm.weight")
    return {"logits": (x @ t("slot_head.weight").t() + t("slot_head.bias")).cpu().numpy()}


def _exact_laya(case, inputs, gguf):
    t, graph = _File(gguf), json.loads(gguf.str("ggmlc.graph_spec"))
    name = {int(i): v["name"] for i, v in graph["tensors"].items()}
    bias, norms, linear_of = {}, {}, {}
    for node in graph["nodes"]:
        ins = node["inputs"]
        if node["opcode"] == 29:  # linear: weight, input[, bias]
            bias[name[ins[0]]] = [name[i] for i in ins[2:]]
            linear_of[node["outputs"][0]] = name[ins[0]]
        elif node["opcode"] == 200 and ins[0] in linear_of:  # a bias added to a linear's output
            bias[linear_of[ins[0]]].append(name[ins[1]])
        elif node["opcode"] == 201:  # layer norm: input[, weight[, bias]]
            norms[node["name"]] = ([name[i] for i in ins[1:]], float(np.float32(node["attributes"]["eps"])))
    gelu = functools.partial(torch.nn.functional.gelu, approximate="tanh")

    def lin(key, x):
        y = x @ t(key + ".weight").view(-1, x.shape[-1]).t()
        return functools.reduce(lambda y, b: y + t(b), bias[key + ".weight"], y)

    def norm(i, x):
        params, eps = norms[f"layer_norm_{i}" if i else "layer_norm"]
        params = [t(p) for p in params] + [None] * (2 - len(params))
        return torch.nn.functional.layer_norm(x, x.shape[-1:], params[0], params[1], eps)

    lengths, n_layers = _lengths(case), case["layers"]
    segments = _segments(lengths)
    tables = {k: (t("cos_" + k), t("sin_" + k)) for k in ("full", "slide")}

    def attention(qkv, kind, window):
        q, k, v = (a.reshape(len(qkv), -1, 64) for a in qkv.chunk(3, -1))
        out = []
        for at, n in zip(segments, lengths):
            qs, ks = q[at], k[at]
            if kind:
                qs, ks = (_rotate(a, tables[kind][0][:n], tables[kind][1][:n], 32) for a in (qs, ks))
            i = torch.arange(n, device=qkv.device)
            out.append(_attend(qs, ks, v[at], (i[:, None] - i[None, :]).abs() <= 64 if window else None))
        return torch.cat(out)

    h = norm(0, t("tok_emb.weight", np.concatenate([ids for ids, _, _ in inputs])))
    for l in range(n_layers):
        x, local = norm(2 * l, h) if l else h, l % 3 != 0
        h = h + lin(f"wo.{l}", attention(lin(f"qkv.{l}", x), "slide" if local else "full", local))
        gate, up = lin(f"mlp_wi.{l}", norm(2 * l + 1, h)).chunk(2, -1)
        h = h + lin(f"mlp_wo.{l}", gelu(gate) * up)
    kinds = torch.as_tensor(np.repeat([q for _, _, q in inputs], lengths), device=h.device)
    h = norm(2 * n_layers, h) + t("type_emb.weight")[kinds]
    for i in range(2):
        j = 2 * n_layers + 1 + 2 * i
        h = h + lin(f"head_wo.{i}", attention(lin(f"head_qkv.{i}", norm(j, h)), None, False))
        h = h + lin(f"head_fc2.{i}", torch.relu(lin(f"head_fc1.{i}", norm(j + 1, h))))
    logits, act = [], []
    for at, (_, markers, _) in zip(segments, inputs):
        z = lin("scorer_fc2", gelu(lin("scorer_fc1", norm(2 * n_layers + 5, h[at][torch.as_tensor(markers, device=h.device).long()]))))[:, 0]
        p, k = torch.softmax(z, 0), max(len(markers), 2)
        top = p.max()
        second = (p * (top - p) / (top - p + 1e-6)).max()
        entropy = -(p * p.clamp_min(1e-9).log()).sum() / math.log(k)
        pooled = torch.cat([h[at.start], torch.stack([top, top - second, entropy, torch.full_like(top, k / 255)])])
        logits.append(z)
        act.append(lin("act_fc2", gelu(lin("act_fc1", pooled[None]))[0]))
    return {"logits": torch.stack(logits).cpu().numpy(), "act": torch.stack(act).cpu().numpy()}


def exact(case, seed):
    if case["call"] == "decode" and case["precision"] != "exact":
        return None  # a rounded cache may turn a near tie, and another token changes all that follows
    gguf = lh.Gguf.from_bytes(lh.SynthImage(case["model"], MODEL_SEED, case["layers"]))
    family = {"openthai-0.8b": _exact_openthai, "laya-english": _exact_laya}.get(case["model"], _exact_decoder)
    with torch.no_grad():
        return family(case, _inputs(case, seed), gguf)

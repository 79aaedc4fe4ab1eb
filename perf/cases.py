"""Timed cases of the forwarder: what a program that serves StableLM- and
Llama-shaped checkpoints calls, from one token to a long prompt.

Kinds of case (each through the public classes of tinyoai_amd.hip):

  product   one weight matrix times n rows on the device
  decode    one token after a resident prefix
  prefill   n tokens after a resident prefix (a prompt, or a chat turn)
  score     n tokens with every position's log probabilities
  branches  a branch session: open, ragged suffixes, lockstep steps, close
  llama     tokens through the stories260K-shaped legacy Llama

Models have few layers and a small vocabulary, so that a layer's work
dominates a pass; every layer of a deep model costs the same.
"""
import math

import numpy as np
import torch

from tinyoai_amd import hip
from tinyoai_amd import weights as W

# Layer shapes: (hidden, heads, kv heads, MLP width).
SHAPES = {"3b": (2560, 32, 32, 6912),     # the benchmark's StableLM-3B shapes
          "clio": (2816, 22, 22, 7552),   # 22 heads of 128
          "gqa": (2048, 32, 8, 5632)}     # grouped-query attention, heads of 64
LLAMA = dict(dim=64, hidden_dim=172, n_layers=5, n_heads=8, n_kv_heads=4, vocab_size=512, seq_len=512)
CONTEXT, THETA, ROTARY, EPS = 8192, 10000.0, 0.25, 1e-5
# Weight formats by name: (MLP and embedding, attention, classifier).
# "kquant" is the usual K-quant mix.
FORMATS = {"q8_0": (W.Q8_0,) * 3, "bf16": (W.BF16,) * 3, "f16": (W.F16,) * 3, "f32": (W.F32,) * 3,
           "q4_k": (W.Q4_K,) * 3, "q5_k": (W.Q5_K,) * 3, "q6_k": (W.Q6_K,) * 3, "q5_1": (W.Q5_1,) * 3,
           "kquant": (W.Q4_K, W.Q6_K, W.Q6_K)}


def listed():
    return [
        # The smallest call: one token of the 260K-parameter story model, bound by launches and latency.
        dict(name="llama_token", kind="llama", prefix=96, n=1, all=False),
        # One weight times one row, as a host that walks the layers itself does for each token.
        dict(name="product_q8_0_row", kind="product", fmt="q8_0", rows=6912, cols=2560, n=1),
        # The same weight times a batch of rows.
        dict(name="product_q8_0_128", kind="product", fmt="q8_0", rows=6912, cols=2560, n=128),
        # A half-precision checkpoint's down projection over a ragged batch.
        dict(name="product_f16_77", kind="product", fmt="f16", rows=2560, cols=6912, n=77),
        # Chat decoding at an ordinary position: quantized weights, fp32 cache.
        dict(name="decode_q8_0", kind="decode", fmt="q8_0", shape="3b", layers=4, vocab=16384, kv=32, prefix=640),
        # Decoding at the end of a long document: BF16 weights, fp16 cache.
        dict(name="decode_bf16_8k", kind="decode", fmt="bf16", shape="3b", layers=4, vocab=16384, kv=16, prefix=8000),
        # A short user turn in a running chat: few tokens after a resident prefix.
        dict(name="turn_q8_0", kind="prefill", fmt="q8_0", shape="3b", layers=2, vocab=4096, kv=32, prefix=430, n=19),
        # The ordinary prompt chunk a host submits.
        dict(name="prompt_q8_0", kind="prefill", fmt="q8_0", shape="3b", layers=2, vocab=4096, kv=32, prefix=0, n=512),
        # A large chunk of a long document, not a multiple of any tile.
        dict(name="prompt_bf16_2k", kind="prefill", fmt="bf16", shape="3b", layers=2, vocab=4096, kv=16, prefix=2048,
             n=1999),
        # A system prompt through a K-quant mix.
        dict(name="prompt_kquant", kind="prefill", fmt="kquant", shape="3b", layers=2, vocab=4096, kv=16, prefix=0,
             n=700),
        # Sixteen continuations of one shared prompt, private suffixes of different lengths, then lockstep tokens.
        dict(name="branches_kquant", kind="branches", fmt="kquant", shape="3b", layers=4, vocab=16384, kv=16,
             prefix=4096, count=16, longest=256, steps=16),
        # Scoring a passage under a half-precision checkpoint: every position against the whole vocabulary.
        dict(name="score_f16", kind="score", fmt="f16", shape="3b", layers=2, vocab=65536, kv=32, prefix=0, n=160,
             top=5),
    ]


def _log(rng, low, high):
    """An integer in [low, high], even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["product", "product", "decode", "decode", "prefill", "prefill", "prefill", "score", "branches",
                       "llama"])
    if kind == "llama":
        prefix = rng.randrange(0, 256)
        return dict(kind=kind, prefix=prefix, n=_log(rng, 1, 255), all=rng.random() < 0.3)
    if kind == "product":
        fmt = rng.choice(["q8_0", "q8_0", "bf16", "f16", "f32", "q4_k", "q5_k", "q6_k", "q5_1"])
        step = {"q8_0": 32, "q5_1": 32, "q4_k": 256, "q5_k": 256, "q6_k": 256}.get(fmt, rng.choice([1, 8, 32]))
        cols = max(1, _log(rng, 512, 8192) // step) * step
        return dict(kind=kind, fmt=fmt, rows=_log(rng, 512, 8192), cols=cols, n=_log(rng, 1, 2048))
    fmt = rng.choice(["q8_0", "q8_0", "bf16", "f16", "kquant", "kquant", "q5_k"])
    shape = rng.choice(["3b", "3b", "gqa"] if fmt in ("kquant", "q5_k") else ["3b", "3b", "clio", "gqa"])
    case = dict(kind=kind, fmt=fmt, shape=shape, layers=2, vocab=rng.choice([4096, 16384]), kv=rng.choice([16, 32]))
    if kind == "decode":
        return dict(case, prefix=_log(rng, 1, 8000))
    if kind == "prefill":
        return dict(case, prefix=rng.choice([0, _log(rng, 16, 4096)]), n=_log(rng, 2, 1999))
    if kind == "score":
        return dict(case, vocab=rng.choice([16384, 32768]), prefix=0, n=_log(rng, 2, 256), top=rng.randint(1, 10))
    return dict(case, vocab=4096, prefix=_log(rng, 64, 4096), count=rng.randint(2, 24), longest=_log(rng, 4, 256),
                steps=rng.randint(8, 16))


# ------------------------------------------------------------ weights
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _half(x):
    """fp16 values and their bytes on a last axis of two."""
    h = x.half()
    return h, h.unsqueeze(-1).view(torch.uint8)


def _matrix(fmt, rows, cols, g, std=0.02):
    """A seeded matrix in its on-disk encoding (uint8 on the GPU) and a function that gives its float64 values:
    normal weights, quantized as a converter would (block scales near their mean, quants over their range)."""
    if fmt in (W.F32, W.F16, W.BF16):
        v = _normal(g, rows, cols) * std
        v = v if fmt == W.F32 else v.half() if fmt == W.F16 else v.bfloat16()
        return v.reshape(-1).view(torch.uint8), lambda: v.double()
    per = 32 if fmt in (W.Q8_0, W.Q5_1) else 256
    nb = rows * cols // per
    spread = 1 + 0.15 * _normal(g, nb, 1).clamp(-3, 3)
    z = _normal(g, nb, per)
    if fmt == W.Q8_0:
        d, db = _half(spread * std * 3 / 127)
        q = (z * (127 / 3)).round().clamp(-127, 127).to(torch.int8)
        raw = torch.cat([db.reshape(nb, 2), q.view(torch.uint8)], 1)
        return raw.reshape(-1), lambda: (d.double() * q.double()).reshape(rows, cols)
    if fmt == W.Q5_1:
        d, db = _half(spread * std * 6 / 31)
        m, mb = _half(-spread * std * 3)
        q = (15.5 + z * 5.2).round().clamp(0, 31).to(torch.uint8)
        bits = ((q >> 4).to(torch.int64) << torch.arange(32, device="cuda")).sum(1)
        high = torch.stack([(bits >> (8 * i)) & 255 for i in range(4)], 1).to(torch.uint8)
        raw = torch.cat([db.reshape(nb, 2), mb.reshape(nb, 2), high, (q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)], 1)
        return raw.reshape(-1), lambda: (d.double() * q.double() + m.double()).reshape(rows, cols)
    if fmt == W.Q6_K:
        sc = torch.randint(24, 121, (nb, 16), generator=g, device="cuda")
        d, db = _half(spread * std / (10 * 72))
        q = (32 + z * 10).round().clamp(0, 63).to(torch.uint8)
        h = q.reshape(nb, 2, 4, 32)  # half, quarter, value
        low = torch.stack([(h[:, :, 0] & 15) | ((h[:, :, 2] & 15) << 4), (h[:, :, 1] & 15) | ((h[:, :, 3] & 15) << 4)], 2)
        top = (h[:, :, 0] >> 4) | ((h[:, :, 1] >> 4) << 2) | ((h[:, :, 2] >> 4) << 4) | ((h[:, :, 3] >> 4) << 6)
        raw = torch.cat([low.reshape(nb, 128), top.reshape(nb, 64), sc.to(torch.uint8), db.reshape(nb, 2)], 1)
        return raw.reshape(-1), lambda: (d.double().reshape(nb, 1, 1) * sc.double().unsqueeze(-1)
                                         * (q.double().reshape(nb, 16, 16) - 32)).reshape(rows, cols)
    five = fmt == W.Q5_K
    mid, wide = (15.5, 6.0) if five else (7.5, 3.0)
    sc = torch.randint(20, 64, (nb, 8), generator=g, device="cuda")
    mn = (sc + torch.randint(-2, 3, (nb, 8), generator=g, device="cuda")).clamp(0, 63)
    d, db = _half(spread * std / (wide * 42))
    m, mb = _half(spread * std / (wide * 42) * mid)
    q = (mid + z * wide).round().clamp(0, 31 if five else 15).to(torch.uint8)
    lo, hi = torch.stack([sc[:, :4], mn[:, :4]], 1), torch.stack([sc[:, 4:], mn[:, 4:]], 1)
    s12 = torch.cat([(lo | ((hi >> 4) << 6)).reshape(nb, 8), (hi[:, 0] & 15) | ((hi[:, 1] & 15) << 4)], 1).to(torch.uint8)
    sub = (q & 15).reshape(nb, 4, 2, 32)
    parts = [db.reshape(nb, 2), mb.reshape(nb, 2), s12]
    if five:
        top = (q >> 4).reshape(nb, 8, 32).to(torch.int64) << torch.arange(8, device="cuda").reshape(1, 8, 1)
        parts.append(top.sum(1).to(torch.uint8))
    raw = torch.cat(parts + [(sub[:, :, 0] | (sub[:, :, 1] << 4)).reshape(nb, 128)], 1)
    return raw.reshape(-1), lambda: (d.double().reshape(nb, 1, 1) * sc.double().unsqueeze(-1)
                                     * q.double().reshape(nb, 8, 32)
                                     - (m.double() * mn.double()).unsqueeze(-1)).reshape(rows, cols)


def _names(case):
    """The model's tensors in the order they are drawn: (name, format or None for a norm, rows, cols)."""
    d, heads, kvh, inter = SHAPES[case["shape"]]
    mlp, att, head = FORMATS[case["fmt"]]
    kv = d // heads * kvh
    yield "model.embed_tokens.weight", mlp, case["vocab"], d
    yield "lm_head.weight", head, case["vocab"], d
    yield "model.norm.weight", None, 1, d
    yield "model.norm.bias", None, 0, d
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        yield p + "input_layernorm.weight", None, 1, d
        yield p + "input_layernorm.bias", None, 0, d
        yield p + "self_attn.q_proj.weight", att, d, d
        yield p + "self_attn.k_proj.weight", att, kv, d
        yield p + "self_attn.v_proj.weight", att, kv, d
        yield p + "self_attn.o_proj.weight", att, d, d
        yield p + "mlp.gate_proj.weight", mlp, inter, d
        yield p + "mlp.up_proj.weight", mlp, inter, d
        yield p + "mlp.down_proj.weight", mlp, d, inter


def _draw_model(case, seed):
    """(name, format, rows, cols, raw bytes, float64 values) of every tensor."""
    g = _gen(seed)
    for name, fmt, rows, cols in _names(case):
        if fmt is None:  # LayerNorm weight about 1, bias about 0
            v = rows + 0.1 * _normal(g, cols)
            yield name, W.F32, 1, cols, v.view(torch.uint8), v.double
        else:
            raw, exact_values = _matrix(fmt, rows, cols, g)
            yield name, fmt, rows, cols, raw, exact_values


def _tokens(case, seed):
    """Every token id the case's calls take, as int32 arrays."""
    r = np.random.default_rng(seed)
    ids = lambda n: r.integers(0, case["vocab"], n).astype(np.int32)  # noqa: E731
    t = {"past": ids(case["prefix"]), "new": ids(case.get("n", 1)), "targets": ids(case.get("n", 1))}
    if case["kind"] == "branches":
        lengths = r.integers(1, case["longest"] + 1, case["count"])
        t["suffixes"] = [ids(n) for n in lengths]
        t["steps"] = [ids(case["count"]) for _ in range(case["steps"])]
    return t


def _llama(seed, prefix, n):
    """A seeded llama2.c payload by name (fp32, scaled as a trained model's) and the token ids."""
    r = np.random.default_rng(seed)
    c, L = LLAMA, LLAMA["n_layers"]
    d, h, hs = c["dim"], c["hidden_dim"], c["dim"] // c["n_heads"]
    kv = hs * c["n_kv_heads"]
    mat = lambda *s: (r.standard_normal(s) * 0.8 / math.sqrt(s[-1])).astype(np.float32)  # noqa: E731
    norm = lambda *s: (1 + 0.1 * r.standard_normal(s)).astype(np.float32)  # noqa: E731
    angle = np.arange(c["seq_len"])[:, None] * 10000.0 ** (-np.arange(0, hs, 2) / hs)
    p = {"emb": mat(c["vocab_size"], d) * np.float32(4), "rms_att": norm(L, d), "wq": mat(L, d, d), "wk": mat(L, kv, d),
         "wv": mat(L, kv, d), "wo": mat(L, d, d), "rms_ffn": norm(L, d), "w1": mat(L, h, d), "w2": mat(L, d, h),
         "w3": mat(L, h, d), "rms_final": norm(d), "cos": np.cos(angle).astype(np.float32),
         "sin": np.sin(angle).astype(np.float32)}
    return p, r.integers(3, c["vocab_size"], prefix + n).astype(np.int32)


# ------------------------------------------------------------ the calls
_stream = []  # the one stream the program runs its products on


def prepare(case, seed):
    kind = case["kind"]
    if kind == "product":
        g = _gen(seed)
        fmt = FORMATS[case["fmt"]][0]
        raw, _ = _matrix(fmt, case["rows"], case["cols"], g)
        x = _normal(g, case["n"], case["cols"])
        y = torch.empty(case["n"], case["rows"], device="cuda")
        torch.cuda.synchronize()
        w = hip.Weight(W.Tensor(fmt, case["rows"], case["cols"], raw.cpu().numpy()))
        if not _stream:
            _stream.append(torch.cuda.Stream())
        return dict(kind=kind, w=w, x=x, y=y, n=case["n"], stream=_stream[0].cuda_stream)
    if kind == "llama":
        p, ids = _llama(seed, case["prefix"], case["n"])
        f = hip.LlamaForwarder(LLAMA, np.concatenate([v.reshape(-1) for v in p.values()]))
        if case["prefix"]:
            f.forward(0, ids[:case["prefix"]])
        return dict(kind=kind, f=f, prefix=case["prefix"], ids=ids[case["prefix"]:], all=case["all"])
    d, heads, kvh, inter = SHAPES[case["shape"]]
    config = dict(W.STABLELM_3B, vocab_size=case["vocab"], hidden_size=d, intermediate_size=inter,
                  num_hidden_layers=case["layers"], num_attention_heads=heads, num_key_value_heads=kvh,
                  max_position_embeddings=CONTEXT, layer_norm_eps=EPS, rope_theta=THETA, partial_rotary_factor=ROTARY)
    tensors = {name: W.Tensor(fmt, rows, cols, raw.cpu().numpy())
               for name, fmt, rows, cols, raw, _ in _draw_model(case, seed)}
    f = hip.StableLMForwarder(config, tensors)
    if case["kv"] == 16:
        f.set_kv_bits(16)
    t = _tokens(case, seed)
    if case["prefix"]:
        f.forward(0, t["past"], want_logits=False)
    state = dict(kind=kind, f=f, prefix=case["prefix"], **t)
    if kind == "score":
        state["top"] = case["top"]
    if kind == "branches":  # the rows of each call, which the program reads between them
        state["rows"] = [np.empty((case["count"], case["vocab"]), np.float32) for _ in range(case["steps"] + 1)]
    torch.cuda.empty_cache()
    return state


def run(s):
    kind = s["kind"]
    if kind == "product":
        s["w"].mul_device(s["x"].data_ptr(), s["n"], s["y"].data_ptr(), s["stream"])
        return s["y"]
    if kind == "llama":
        return s["f"].forward(s["prefix"], s["ids"], s["all"])
    if kind == "score":
        logits, chosen, ids, logprobs = s["f"].forward_with_logprobs(s["prefix"], s["new"], s["targets"], s["top"])
        return dict(logits=logits, chosen=chosen, ids=ids, logprobs=logprobs)
    if kind == "branches":
        b = s["f"].new_branches(s["prefix"], len(s["suffixes"]))
        b.append(s["suffixes"], out=s["rows"][0])
        for tokens, out in zip(s["steps"], s["rows"][1:]):
            b.forward(tokens, out=out)
        b.close()
        return s["rows"]
    return s["f"].forward(s["prefix"], s["new"])


# ------------------------------------------------------------ what a pass costs
def _parameters(case):
    """(values, bytes) of the layers' matrices, and of the classifier."""
    layers, head = [0, 0], [0, 0]
    for name, fmt, rows, cols in _names(case):
        if fmt is not None and not name.startswith("model.embed"):
            to = head if name.startswith("lm_head") else layers
            to[0] += rows * cols
            to[1] += W.nbytes(fmt, rows, cols)
    return layers, head


def work(case):
    if case["kind"] == "product":
        rows, cols, n = case["rows"], case["cols"], case["n"]
        return {"bytes": W.nbytes(FORMATS[case["fmt"]][0], rows, cols) + 4 * n * (rows + cols),
                "flops": 2 * n * rows * cols}
    if case["kind"] == "llama":
        c, n, p = LLAMA, case["n"], case["prefix"]
        kv = c["dim"] // c["n_heads"] * c["n_kv_heads"]
        layer = c["dim"] * (2 * c["dim"] + 2 * kv + 3 * c["hidden_dim"])
        rows, head = (n if case["all"] else 1), c["vocab_size"] * c["dim"]
        return {"bytes": 4 * (c["n_layers"] * (layer + 2 * kv * (p + 2 * n)) + head + rows * c["vocab_size"]),
                "flops": 2 * n * c["n_layers"] * layer + 2 * rows * head
                + 4 * c["dim"] * c["n_layers"] * (n * p + n * (n + 1) // 2)}
    d, heads, kvh, _ = SHAPES[case["shape"]]
    (values, nbytes), (hvalues, hbytes) = _parameters(case)
    L, p, kvb = case["layers"], case["prefix"], 2 * (d // heads * kvh) * case["kv"] // 8
    if case["kind"] == "branches":
        t = _tokens(case, 0)
        total = {"bytes": 0, "flops": 0}
        long = [len(x) for x in t["suffixes"]]
        for step in range(case["steps"] + 1):  # the append, then each lockstep step
            new = long if step == 0 else [1] * len(long)
            past = [0] * len(long) if step == 0 else [x + step - 1 for x in long]
            n = sum(new)
            total["bytes"] += nbytes + hbytes + 4 * len(long) * case["vocab"] + L * kvb * (p + sum(past) + n)
            total["flops"] += 2 * n * values + 2 * len(long) * hvalues
            total["flops"] += sum(4 * d * L * (k * (p + q) + k * (k + 1) // 2) for k, q in zip(new, past))
        return total
    n = case.get("n", 1)
    rows = n if case["kind"] == "score" else 1
    return {"bytes": nbytes + hbytes + 4 * case["vocab"] + L * kvb * (p + n),
            "flops": 2 * n * values + 2 * rows * hvalues + 4 * d * L * (n * p + n * (n + 1) // 2)}


def tolerance(case):
    """About four times the error against float64 measured for each kind: fp32 sums; activations of 16 significant bits
    in the matrix-core products of Q8_0 and BF16 weights; an fp16 cache, whose keys and values (and the queries and
    softmax weights beside them) are rounded to 11 bits."""
    if case["kind"] == "llama":
        return {"rel": 2e-6}
    planes = case["fmt"] in ("q8_0", "bf16")
    if case["kind"] == "product":
        return {"rel": 1e-5 if planes and case["n"] > 1 else 2e-6}
    rel = 5e-4 if case["kv"] == 16 else 3e-5 if planes else 5e-6
    return {"rel": rel, "differ": 0.01 if case["kv"] == 16 else 0.002} if case["kind"] == "score" else {"rel": rel}


# ------------------------------------------------------------ 64 bits
def _llama64(case, seed):
    p, ids = _llama(seed, case["prefix"], case["n"])
    p = {k: torch.from_numpy(v).double() for k, v in p.items()}
    c = LLAMA
    hs, kvh = c["dim"] // c["n_heads"], c["n_kv_heads"]
    n = len(ids)
    cos, sin = p["cos"][:n, None], p["sin"][:n, None]
    scale = float(np.sqrt(np.float32(hs)))
    norm = lambda x, w: x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt() * w  # noqa: E731

    def turn(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    x = p["emb"][torch.from_numpy(ids).long()]
    mask = torch.ones(n, n, dtype=torch.bool).tril()
    for i in range(c["n_layers"]):
        h = norm(x, p["rms_att"][i])
        q = turn((h @ p["wq"][i].T).reshape(n, -1, hs))
        k = turn((h @ p["wk"][i].T).reshape(n, -1, hs)).repeat_interleave(c["n_heads"] // kvh, 1)
        v = (h @ p["wv"][i].T).reshape(n, -1, hs).repeat_interleave(c["n_heads"] // kvh, 1)
        s = torch.einsum("qhd,khd->hqk", q, k) / scale
        a = s.masked_fill(~mask, -math.inf).softmax(-1)
        x = x + torch.einsum("hqk,khd->qhd", a, v).reshape(n, -1) @ p["wo"][i].T
        h = norm(x, p["rms_ffn"][i])
        x = x + (torch.nn.functional.silu(h @ p["w1"][i].T) * (h @ p["w3"][i].T)) @ p["w2"][i].T
    rows = norm(x[case["prefix"]:] if case["all"] else x[-1:], p["rms_final"]) @ p["emb"].T
    return rows if case["all"] else rows[0]


class _Stable64:
    """The StableLM block in float64, with a cache of its keys and values (rounded to fp16 where the cache is)."""

    def __init__(self, case, seed):
        self.c = case
        self.t = {name: v().reshape(rows, cols) if rows > 1 else v().reshape(-1)
                  for name, _, rows, cols, _, v in _draw_model(case, seed)}
        d, self.heads, self.kvh, _ = SHAPES[case["shape"]]
        self.hd = d // self.heads
        rot = int(self.hd * ROTARY)
        # the rotation's angles are float32 products of the position and the frequency
        power = np.array([np.float32(THETA ** float(np.float32(2 * i) / np.float32(rot))) for i in range(rot // 2)])
        angle = (np.arange(CONTEXT, dtype=np.float32)[:, None] * (np.float32(1) / power)[None]).astype(np.float64)
        self.rot = rot
        self.cos, self.sin = (torch.from_numpy(f(angle).astype(np.float32)).double().cuda() for f in (np.cos, np.sin))

    def _norm(self, x, p):
        x = x - x.mean(-1, keepdim=True)
        return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * self.t[p + ".weight"] + self.t[p + ".bias"]

    def _turn(self, x, pos):
        r = self.rot // 2
        a, b, c, s = x[..., :r], x[..., r:self.rot], self.cos[pos][:, None], self.sin[pos][:, None]
        return torch.cat([a * c - b * s, b * c + a * s, x[..., self.rot:]], -1)

    def rows(self, ids, past):
        """The residual stream of `ids` after the cache `past` (a list of (k, v) per layer), and the longer cache."""
        t, hd = self.t, self.hd
        n, start = len(ids), (past[0][0].shape[1] if past else 0)
        pos = torch.arange(start, start + n, device="cuda")
        x = t["model.embed_tokens.weight"][torch.from_numpy(np.asarray(ids)).long().cuda()]
        scale, grown = float(np.sqrt(np.float32(hd))), []
        for i in range(self.c["layers"]):
            p = f"model.layers.{i}."
            h = self._norm(x, p + "input_layernorm")
            q, k, v = ((h @ t[p + f"self_attn.{w}_proj.weight"].T).reshape(n, -1, hd) for w in "qkv")
            q, k = self._turn(q, pos).transpose(0, 1), self._turn(k, pos).transpose(0, 1)
            v = v.transpose(0, 1)
            if self.c["kv"] == 16:
                k, v = k.half().double(), v.half().double()
            if past:
                k, v = torch.cat([past[i][0], k], 1), torch.cat([past[i][1], v], 1)
            grown.append((k, v))
            out = torch.empty(n, self.heads, hd, dtype=torch.float64, device="cuda")
            for head in range(self.heads):
                kk, vv = (y[head * self.kvh // self.heads].contiguous() for y in (k, v))
                for r0 in range(0, n, 2048):
                    s = q[head, r0:r0 + 2048].contiguous() @ kk.T.contiguous() / scale
                    late = torch.arange(k.shape[1], device="cuda")[None] > pos[r0:r0 + 2048, None]
                    out[r0:r0 + 2048, head] = s.masked_fill_(late, -math.inf).softmax(-1) @ vv
            gate = torch.nn.functional.silu(h @ t[p + "mlp.gate_proj.weight"].T) * (h @ t[p + "mlp.up_proj.weight"].T)
            x = x + out.reshape(n, -1) @ t[p + "self_attn.o_proj.weight"].T + gate @ t[p + "mlp.down_proj.weight"].T
        return x, grown

    def logits(self, x):
        return self._norm(x, "model.norm") @ self.t["lm_head.weight"].T


def exact(case, seed):
    if case["kind"] == "product":
        g = _gen(seed)
        _, values = _matrix(FORMATS[case["fmt"]][0], case["rows"], case["cols"], g)
        return _normal(g, case["n"], case["cols"]).double() @ values().T
    if case["kind"] == "llama":
        return _llama64(case, seed)
    m, t = _Stable64(case, seed), _tokens(case, seed)
    past = m.rows(t["past"], None)[1] if case["prefix"] else None
    if case["kind"] == "branches":
        got = [[] for _ in range(case["steps"] + 1)]
        for j, suffix in enumerate(t["suffixes"]):
            ids = np.concatenate([suffix, [s[j] for s in t["steps"]]])
            rows = m.logits(m.rows(ids, past)[0][len(suffix) - 1:])
            for k in range(case["steps"] + 1):
                got[k].append(rows[k].cpu())
        return [torch.stack(rows) for rows in got]
    x, _ = m.rows(t["new"], past)
    if case["kind"] == "score":
        lp = m.logits(x)
        logits = lp[-1].clone()
        lp -= lp.logsumexp(-1, keepdim=True)
        top = lp.topk(case["top"], -1)
        chosen = lp[torch.arange(len(lp), device="cuda"), torch.from_numpy(t["targets"]).long().cuda()]
        return dict(logits=logits, chosen=chosen, ids=None, logprobs=top.values)
    return m.logits(x[-1:])[0]

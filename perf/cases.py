"""The work whose speed is measured: calls that a user of the framework makes, through its public
entry points, over the range of sizes, weight formats and directions that real use has.

Three levels.  The operator level (GpuWeightTensor.mat_mul and the attention, sampling, norm and
block-codec operators) is what a host that keeps its own forward pass calls.  The model level
(GpuTransformerModel, GpuInferenceSession) is what a server or a command-line program calls:
prompt prefill, token-by-token decode and lockstep decode of many sessions.  Sizes are those of
synthetic.WORKLOADS and synthetic.GEMV_SHAPES (GPT-2 small, a 1.1B and a 1.7B LLaMA-style
model) and, in draw(), generic ones between them.
"""
import math

import numpy as np
import torch

from smallmind_amd import quantization as Q
from smallmind_amd.model import GpuInferenceSession, GpuTransformerModel, ModelConfig

TYPES = {"q4_0": 2, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}


def listed():
    return [
        # one projection of a small model for one new token: the smallest call of a decode step,
        # where the launch counts and not the bytes (GPT-2 small's fused QKV)
        {"name": "linear decode q8_0 small", "kind": "linear", "type": "q8_0", "m": 1, "n": 2304, "k": 768},
        # the widest layer matrix of a 1.1B model for one new token: what token-by-token decode
        # streams most bytes from
        {"name": "linear decode q4_k gate/up", "kind": "linear", "type": "q4_k", "m": 1, "n": 11264, "k": 2048},
        # a layer matrix for one token of each of 16 sessions: a step of a serving batch
        {"name": "linear batch q5_k down", "kind": "linear", "type": "q5_k", "m": 16, "n": 2048, "k": 8192},
        # a layer matrix over an ordinary prompt (ragged: 511 tokens before the last one)
        {"name": "linear prompt q4_k gate/up", "kind": "linear", "type": "q4_k", "m": 511, "n": 11264, "k": 2048},
        # a layer matrix over a chunk of a long prompt: the largest single operator call
        {"name": "linear long prompt q8_0 down", "kind": "linear", "type": "q8_0", "m": 2048, "n": 2048, "k": 5632},
        # attention of one new token at an ordinary context, grouped-query heads
        {"name": "attention decode", "kind": "attention_decode", "heads": 32, "kv_heads": 4, "hd": 64, "n_pos": 700,
         "ctx": 768},
        # attention of a chunk of a long prompt over the chunks before it
        {"name": "attention long prompt", "kind": "attention_prefill", "heads": 32, "kv_heads": 4, "hd": 64,
         "p_first": 2048, "m": 2048},
        # next-token sampling with the usual options over a 32000-token vocabulary, after every
        # token of a sampled generation
        {"name": "sample", "kind": "sample", "n": 32000, "context": 300, "temperature": 0.8, "top_k": 40,
         "top_p": 0.95, "min_p": 0.05, "repetition": 1.1},
        # encoding a layer matrix and decoding it again: model import and export
        {"name": "codec q4_k", "kind": "codec", "type": "q4_k", "n": 5632 * 2048},
        # a user's request to a 1.1B chat model: a 512-token prompt and 128 greedy tokens
        {"name": "generate 1.1B q4_k", "kind": "generate", "arch": "llama", "vocab": 32000, "d": 2048, "layers": 22,
         "heads": 32, "kv_heads": 4, "ff": 5632, "type": "q4_k", "embd": "q6_k", "tied": False, "sessions": 1,
         "prompt": 512, "new": 128},
        # a long document read by the same model in 8 bits: a 4096-token prompt, its logits
        {"name": "prefill 1.1B q8_0 4k", "kind": "prefill", "arch": "llama", "vocab": 32000, "d": 2048, "layers": 22,
         "heads": 32, "kv_heads": 4, "ff": 5632, "type": "q8_0", "embd": "q6_k", "tied": False, "prompt": 4096},
        # 16 requests served together by a 1.7B model: 256-token prompts, 64 tokens each
        {"name": "serve 16 x 1.7B q5_k", "kind": "generate", "arch": "llama", "vocab": 49152, "d": 2048,
         "layers": 24, "heads": 32, "kv_heads": 32, "ff": 8192, "type": "q5_k", "embd": "q5_k", "tied": True,
         "sessions": 16, "prompt": 256, "new": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "attention_decode", "attention_prefill", "sample", "codec",
                       "norm", "generate", "prefill"])
    if kind == "linear":
        t = rng.choice(sorted(TYPES))
        k = 256 * _log(rng, 2, 43)
        n = _log(rng, 300, 16384)
        most = 2048 * 2048 * 5632 / (n * k)          # no more products than the largest listed one
        m = max(1, min(_log(rng, 1, 2048), int(most)))
        return {"kind": kind, "type": t, "m": m, "n": n, "k": k}
    if kind == "attention_decode":
        hq, hk = rng.choice([(12, 12), (32, 4), (32, 8), (32, 32)])
        p = _log(rng, 16, 4200)
        return {"kind": kind, "heads": hq, "kv_heads": hk, "hd": rng.choice([64, 64, 128]), "n_pos": p,
                "ctx": (p + rng.randrange(1, 200) + 3) // 4 * 4}
    if kind == "attention_prefill":
        hq, hk = rng.choice([(12, 12), (32, 4), (32, 8), (32, 32)])
        return {"kind": kind, "heads": hq, "kv_heads": hk, "hd": 64, "p_first": rng.choice([0, _log(rng, 16, 2048)]),
                "m": _log(rng, 9, 2048)}
    if kind == "sample":
        return {"kind": kind, "n": _log(rng, 1000, 50257), "context": _log(rng, 8, 2000),
                "temperature": round(rng.uniform(0.6, 1.2), 2), "top_k": rng.choice([0, 20, 40, 100]),
                "top_p": rng.choice([0.8, 0.9, 0.95, 1.0]), "min_p": rng.choice([0.0, 0.05]),
                "repetition": rng.choice([1.0, 1.1])}
    if kind == "codec":
        return {"kind": kind, "type": rng.choice(sorted(TYPES)), "n": 256 * _log(rng, 64, 45056)}
    if kind == "norm":
        return {"kind": kind, "layer": rng.random() < 0.5, "m": _log(rng, 1, 2048), "n": 4 * _log(rng, 64, 2048)}
    arch = rng.choice(["llama", "gpt2"])
    t = rng.choice(["q4_0", "q8_0", "q4_k", "q5_k", "q6_k"])
    if arch == "gpt2":
        d, ff, hq, hk = 768, 3072, 12, 12
    else:
        d, ff, hq, hk = rng.choice([(1024, 2816, 16, 4), (2048, 5632, 32, 4), (2048, 8192, 32, 32)])
    c = {"kind": kind, "arch": arch, "vocab": rng.randrange(16000, 50257), "d": d, "layers": rng.randrange(2, 7),
         "heads": hq, "kv_heads": hk, "ff": ff, "type": t, "embd": t, "tied": True, "prompt": _log(rng, 9, 900)}
    if kind == "generate":
        c["sessions"] = rng.choice([1, 1, _log(rng, 2, 24)])
        c["new"] = _log(rng, 8, 100)
    return c


# ---- weight blocks, written and read here in plain torch ---------------------------------------
def _gen(seed, i=0):
    return torch.Generator(device="cuda").manual_seed(seed * 100003 + i * 7919 + 1)


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8).reshape(*x.shape, 2)


def _pack6(v):
    """[..., 8] six-bit values -> [..., 6] bytes, lowest bits first."""
    a = torch.zeros(v.shape[:-1], dtype=torch.int64, device=v.device)
    for j in range(8):
        a |= v[..., j].to(torch.int64) << (6 * j)
    return torch.stack([(a >> (8 * i)) & 255 for i in range(6)], -1).to(torch.uint8)


def _unpack6(b):
    a = torch.zeros(b.shape[:-1], dtype=torch.int64, device=b.device)
    for i in range(6):
        a |= b[..., i].to(torch.int64) << (8 * i)
    return torch.stack([(a >> (6 * j)) & 63 for j in range(8)], -1)


def _nibbles(q):
    return (q[..., 0::2] | (q[..., 1::2] << 4)).to(torch.uint8)


def _codes(shape, g, mean, std, lo, hi):
    x = torch.empty(shape, dtype=torch.float16, device="cuda").normal_(mean, std, generator=g)
    return x.round_().clamp_(lo, hi).to(torch.int16)


def make_blocks(t, n, g, std):
    """n weights of about N(0, std) as blocks of format t: bell-shaped codes, scales that differ from
    block to block as a quantizer's do."""
    be, _ = BLOCK[t]
    nb = n // be
    vary = lambda *s: 0.7 + 0.6 * torch.rand(*s, device="cuda", generator=g)  # noqa: E731
    if t == "q8_0":
        q = _codes((nb, 32), g, 0.0, 42.0, -127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_f16_bytes(vary(nb) * (std / 42)), q], 1).reshape(-1)
    if t == "q4_0":
        q = _codes((nb, 32), g, 0.0, 2.6, -8, 7) & 15
        return torch.cat([_f16_bytes(vary(nb) * (std / 2.6)), _nibbles(q)], 1).reshape(-1)
    if t in ("q4_k", "q5_k"):
        sc = torch.randint(32, 64, (nb, 8), device="cuda", generator=g)
        if t == "q4_k":
            q = _codes((nb, 256), g, 7.5, 2.6, 0, 15)
            d = vary(nb) * (std / (2.6 * 47))
            return torch.cat([_f16_bytes(d), _f16_bytes(7.5 * d), _pack6(sc), _pack6(sc), _nibbles(q)], 1).reshape(-1)
        q = _codes((nb, 256), g, 16.0, 5.2, 0, 31)
        d = vary(nb) * (std / (5.2 * 47))
        mn = torch.randint(0, 4, (nb, 8), device="cuda", generator=g)
        hb = (q >> 4).reshape(nb, 32, 8)
        qh = sum(hb[..., i] << i for i in range(8)).to(torch.uint8)
        return torch.cat([_f16_bytes(d), _f16_bytes(0.5 * d), _pack6(sc), _pack6(mn), qh, _nibbles(q & 15)],
                         1).reshape(-1)
    q = _codes((nb, 256), g, 32.0, 10.0, 0, 63)
    sc = torch.randint(64, 128, (nb, 16), device="cuda", generator=g).to(torch.int8).view(torch.uint8)
    h = (q >> 4).reshape(nb, 64, 4)
    qh = sum(h[..., i] << (2 * i) for i in range(4)).to(torch.uint8)
    return torch.cat([_nibbles(q & 15), qh, sc, _f16_bytes(vary(nb) * (std / (10 * 96)))], 1).reshape(-1)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _both(b):
    b = b.to(torch.int64)
    return torch.stack([b & 15, b >> 4], -1).reshape(b.shape[0], -1)


def read_blocks(t, blocks):
    """The weights that blocks of format t hold, in 64 bits."""
    be, nbytes = BLOCK[t]
    b = blocks.reshape(-1, nbytes)
    if t == "q8_0":
        return (b[:, 2:].contiguous().view(torch.int8).double() * _half(b[:, :2])).reshape(-1)
    if t == "q4_0":
        q = _both(b[:, 2:])
        return (torch.where(q < 8, q, q - 16).double() * _half(b[:, :2])).reshape(-1)
    if t in ("q4_k", "q5_k"):
        q = _both(b[:, 16:] if t == "q4_k" else b[:, 48:])
        if t == "q5_k":
            bits = torch.arange(8, device=b.device)
            q = q + (((b[:, 16:48].to(torch.int64)[..., None] >> bits) & 1).reshape(-1, 256) << 4) - 16
        sc = (_half(b[:, :2]) * _unpack6(b[:, 4:10])).repeat_interleave(32, 1)
        mn = (_half(b[:, 2:4]) * _unpack6(b[:, 10:16])).repeat_interleave(32, 1)
        return (sc * q - mn).reshape(-1)
    bits = 2 * torch.arange(4, device=b.device)
    q = _both(b[:, :128]) + (((b[:, 128:192].to(torch.int64)[..., None] >> bits) & 3).reshape(-1, 256) << 4) - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1)
    return (sc * q * _half(b[:, 208:])).reshape(-1)


# ---- states --------------------------------------------------------------------------------------
def _acts(m, k, g):
    """Activations as they leave a norm: about unit size, a few features several times larger."""
    x = torch.randn(m, k, device="cuda", generator=g)
    f = torch.ones(k, device="cuda")
    f[torch.randint(0, k, (max(1, k // 100),), device="cuda", generator=g)] = 6.0
    return x * f


def _kv(c, n_pos, ctx, g):
    k = torch.randn(c["kv_heads"], c["hd"], ctx, device="cuda", generator=g)
    v = torch.randn(c["kv_heads"], ctx, c["hd"], device="cuda", generator=g)
    return k, v


class Model:
    """A loaded model with its sessions and requests, closed with the object."""

    def __init__(self, c, seed):
        ctx = -(-(c["prompt"] + c.get("new", 0) + 1) // 16) * 16
        gpt2 = c["arch"] == "gpt2"
        d, ff, kv, V = c["d"], c["ff"], c["d"] // c["heads"] * c["kv_heads"], c["vocab"]
        self.model = GpuTransformerModel(ModelConfig(c["arch"], V, ctx, d, c["layers"], c["heads"], c["kv_heads"], ff))
        g = _gen(seed)
        ones, zeros = torch.ones(max(d, ff), device="cuda"), torch.zeros(max(d, ff), device="cuda")

        def put(name, t, k, n, std):
            self.model.load_tensor(name, TYPES[t], (k, n), make_blocks(t, k * n, g, std))

        def vec(name, n, kind):
            v = {"g": ones, "0": zeros}[kind][:n] if kind in "g0" else torch.randn(n, device="cuda", generator=g) * 0.02
            self.model.load_tensor(name, 0, (n,), v.contiguous())

        # embeddings large enough that a token's own row stands out in a tied head, as a trained
        # model's next token stands out: the greedy choice is then no near-tie
        put("token_embd.weight", c["embd"], d, V, 0.3)
        if gpt2:
            put("position_embd.weight", c["embd"], d, ctx, 0.02)
        for i in range(c["layers"]):
            p = "blk.%d." % i
            vec(p + "attn_norm.weight", d, "g")
            vec(p + "ffn_norm.weight", d, "g")
            if gpt2:
                put(p + "attn_qkv.weight", c["type"], d, d + 2 * kv, 0.02)
                put(p + "ffn_up.weight", c["type"], d, ff, 0.02)
                for name, n, kind in (("attn_norm.bias", d, "0"), ("ffn_norm.bias", d, "0"),
                                      ("attn_qkv.bias", d + 2 * kv, "b"), ("attn_output.bias", d, "b"),
                                      ("ffn_up.bias", ff, "b"), ("ffn_down.bias", d, "b")):
                    vec(p + name, n, kind)
            else:
                for name, n in (("attn_q", d), ("attn_k", kv), ("attn_v", kv), ("ffn_gate", ff), ("ffn_up", ff)):
                    put(p + name + ".weight", c["type"], d, n, 0.02)
            put(p + "attn_output.weight", c["type"], d, d, 0.02)
            put(p + "ffn_down.weight", c["type"], ff, d, 0.02)
        vec("output_norm.weight", d, "g")
        if gpt2:
            vec("output_norm.bias", d, "0")
        if not c["tied"]:
            # the same blocks as the embedding: an untied matrix, read by itself
            gh = _gen(seed)
            self.model.load_tensor("output.weight", TYPES[c["embd"]], (d, V), make_blocks(c["embd"], d * V, gh, 0.3))
        self.model.finalize()
        self.sessions = [self.model.create_session(ctx) for _ in range(c.get("sessions", 1))]
        r = np.random.default_rng(seed)
        self.prompts = [r.integers(0, V, c["prompt"]).astype(np.int32) for _ in self.sessions]
        self.new = c.get("new", 0)

    def __del__(self):
        if getattr(self, "model", None) is not None:
            torch.cuda.synchronize()
            self.model.close()


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "linear":
        blocks = make_blocks(c["type"], c["n"] * c["k"], g, 0.02)
        return {"case": c, "x": _acts(c["m"], c["k"], g), "out": torch.empty(c["m"], c["n"], device="cuda"),
                "w": Q.GpuWeightTensor(TYPES[c["type"]], c["n"], c["k"], blocks)}
    if kind == "attention_decode":
        q = torch.randn(c["heads"] * c["hd"], device="cuda", generator=g)
        k, v = _kv(c, c["n_pos"], c["ctx"], g)
        return {"case": c, "q": q, "k": k, "v": v}
    if kind == "attention_prefill":
        q = torch.randn(c["m"], c["heads"], c["hd"], device="cuda", generator=g)
        k, v = _kv(c, c["p_first"] + c["m"], _prefill_ctx(c), g)
        return {"case": c, "q": q, "k": k, "v": v}
    if kind == "sample":
        return {"case": c, "logits": torch.randn(c["n"], device="cuda", generator=g) * 3.0,
                "ctx": torch.randint(0, c["n"], (c["context"],), device="cuda", generator=g, dtype=torch.int32),
                "u": float(np.random.default_rng(seed).random())}
    if kind == "codec":
        return {"case": c, "x": torch.randn(c["n"], device="cuda", generator=g) * 0.02}
    if kind == "norm":
        return {"case": c, "x": _acts(c["m"], c["n"], g), "g": 1.0 + 0.1 * torch.randn(c["n"], device="cuda", generator=g),
                "b": 0.1 * torch.randn(c["n"], device="cuda", generator=g)}
    return {"case": c, "model": Model(c, seed)}


def _prefill_ctx(c):
    return (c["p_first"] + c["m"] + 3) // 4 * 4


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear":
        return state["w"].mat_mul(state["x"], state["out"], c["m"], c["k"], c["n"])
    if kind == "attention_decode":
        return Q.attention_decode(state["q"], state["k"], state["v"], c["heads"], c["kv_heads"], c["hd"], c["ctx"],
                                  c["n_pos"])
    if kind == "attention_prefill":
        return Q.attention_prefill(state["q"], state["k"], state["v"], c["heads"], c["kv_heads"], c["hd"],
                                   _prefill_ctx(c), c["p_first"], c["m"])
    if kind == "sample":
        return Q.sample(state["logits"], state["u"], state["ctx"], temperature=c["temperature"], top_k=c["top_k"],
                        top_p=c["top_p"], min_p=c["min_p"], repetition_penalty=c["repetition"])
    if kind == "codec":
        blocks = Q.quantize(TYPES[c["type"]], state["x"])
        return blocks, Q.dequantize(TYPES[c["type"]], blocks, c["n"])
    if kind == "norm":
        if c["layer"]:
            return Q.layernorm(state["x"], state["g"], state["b"])
        return Q.rmsnorm(state["x"], state["g"])
    m = state["model"]
    if kind == "prefill":
        return m.sessions[0].forward(m.prompts[0], 0)
    # generated tokens, then the logits that follow the last of them
    if len(m.sessions) == 1:
        toks, _ = m.sessions[0].generate_greedy(m.prompts[0], m.new)
        return toks, m.sessions[0].forward(toks[-1:], c["prompt"] + m.new - 1)
    toks, _ = GpuInferenceSession.generate_greedy_batch(m.sessions, m.prompts, m.new)
    return toks, [s.forward(toks[i, -1:], c["prompt"] + m.new - 1) for i, s in enumerate(m.sessions)]


# ---- what a pass cannot do without ---------------------------------------------------------------
def _mat_bytes(t, n, k):
    be, nbytes = BLOCK[t]
    return n * k // be * nbytes


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": _mat_bytes(c["type"], n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "attention_decode":
        hd, p = c["hd"], c["n_pos"]
        return {"bytes": 4 * (2 * c["kv_heads"] * p * hd + 2 * c["heads"] * hd), "flops": 4 * c["heads"] * p * hd}
    if kind == "attention_prefill":
        hd, m = c["hd"], c["m"]
        pairs = m * c["p_first"] + m * (m + 1) // 2
        return {"bytes": 4 * (2 * c["kv_heads"] * (c["p_first"] + m) * hd + 2 * m * c["heads"] * hd),
                "flops": 4 * c["heads"] * pairs * hd}
    if kind == "sample":
        return {"bytes": 8 * c["n"] + 4 * c["context"], "flops": 10 * c["n"]}
    if kind == "codec":
        b = _mat_bytes(c["type"], 1, c["n"])
        return {"bytes": 8 * c["n"] + 2 * b, "flops": 8 * c["n"]}
    if kind == "norm":
        return {"bytes": 8 * c["m"] * c["n"] + 8 * c["n"], "flops": 6 * c["m"] * c["n"]}
    d, ff, kv, L = c["d"], c["ff"], c["d"] // c["heads"] * c["kv_heads"], c["layers"]
    up = ff if c["arch"] == "gpt2" else 2 * ff
    mats = [(d + 2 * kv, d), (d, d), (up, d), (d, ff)]
    layer_bytes = L * sum(_mat_bytes(c["type"], n, k) for n, k in mats)
    layer_ops = 2 * L * sum(n * k for n, k in mats)
    head_bytes, head_ops = _mat_bytes(c["embd"], c["vocab"], d), 2 * c["vocab"] * d
    s, p, new = c.get("sessions", 1), c["prompt"], c.get("new", 0)
    kv_pos = 8 * L * kv                                   # K and V bytes of one position
    if kind == "prefill":
        return {"bytes": layer_bytes + head_bytes + kv_pos * p + 4 * c["vocab"],
                "flops": p * layer_ops + head_ops + 2 * L * p * p * d}
    steps = new + 1                                       # the generated tokens and the logits after them
    read = sum(p + i for i in range(steps))
    return {"bytes": layer_bytes + steps * (layer_bytes + head_bytes) + s * kv_pos * (p + read),
            "flops": s * ((p + steps) * layer_ops + steps * head_ops + 2 * L * p * p * d + 4 * L * read * d)}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # 32-bit sums of up to 11008 terms; measured against 64 bits: 3e-7 (one row) to 5.3e-6
        # (many rows of a format whose blocks carry an offset)
        return {"rel": 2e-5, "max": 2e-4}
    if kind in ("attention_decode", "attention_prefill"):
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "sample":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "codec":
        return "exact"
    if kind == "norm":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 2e-4, "max": 2e-3, "differ": 0.01}


# ---- the same in 64 bits -------------------------------------------------------------------------
def _fast_exp(x):
    """The Pade [2/2] exponential that the reference's softmax uses."""
    x = x.clamp(-87.3, 88.7)
    h, q = x * 0.5, x * x * 0.08333333
    return (1 + h + q) / (1 - h + q)


def exact(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "linear":
        w = read_blocks(c["type"], make_blocks(c["type"], c["n"] * c["k"], g, 0.02)).reshape(c["n"], c["k"])
        return _acts(c["m"], c["k"], g).double() @ w.t()
    if kind == "attention_decode":
        q = torch.randn(c["heads"] * c["hd"], device="cuda", generator=g).double().reshape(c["heads"], 1, c["hd"])
        k, v = _kv(c, c["n_pos"], c["ctx"], g)
        return _attend(c, q, k, v, c["n_pos"] - 1).reshape(-1)
    if kind == "attention_prefill":
        q = torch.randn(c["m"], c["heads"], c["hd"], device="cuda", generator=g).double()
        k, v = _kv(c, c["p_first"] + c["m"], _prefill_ctx(c), g)
        return _attend(c, q.transpose(0, 1), k, v, c["p_first"]).transpose(0, 1).reshape(-1)
    if kind == "sample":
        return [None, _sample(c, torch.randn(c["n"], device="cuda", generator=g) * 3.0, g)]
    if kind == "norm":
        x = _acts(c["m"], c["n"], g).double()
        ga = (1.0 + 0.1 * torch.randn(c["n"], device="cuda", generator=g)).double()
        be = (0.1 * torch.randn(c["n"], device="cuda", generator=g)).double()
        if c["layer"]:
            x = x - x.mean(1, keepdim=True)
        y = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * ga
        return y + be if c["layer"] else y
    return None


def _attend(c, q, k, v, p_first):
    """q [heads][m][hd] at positions p_first ...: [heads][m][hd]."""
    G, m = c["heads"] // c["kv_heads"], q.shape[1]
    out = []
    for h in range(c["heads"]):
        n = p_first + m
        kh, vh = k[h // G, :, :n].double(), v[h // G, :n].double()
        s = (q[h] @ kh) / math.sqrt(c["hd"])
        seen = torch.arange(n, device="cuda")[None, :] <= p_first + torch.arange(m, device="cuda")[:, None]
        s = s.masked_fill(~seen, -math.inf)
        e = torch.where(seen, _fast_exp(s - s.amax(1, keepdim=True)), 0.0)
        out.append(e @ vh / e.sum(1, keepdim=True))
    return torch.stack(out)


def _sample(c, logits, g):
    ctx = torch.randint(0, c["n"], (c["context"],), device="cuda", generator=g, dtype=torch.int32)
    lg = logits.double()
    if c["repetition"] != 1.0:
        t = ctx[max(0, c["context"] - min(c["context"], 256)):].unique().long()
        r = float(np.float32(c["repetition"]))
        lg[t] = torch.where(lg[t] > 0, lg[t] / r, lg[t] * r)
    lg = lg / float(np.float32(c["temperature"]))
    if 0 < c["top_k"] < c["n"]:
        lg = torch.where(lg >= lg.topk(c["top_k"]).values[-1], lg, -math.inf)
    p = torch.softmax(lg, 0)
    if c["top_p"] < 1.0:
        s, order = p.sort(descending=True)
        keep = s.cumsum(0) - s < c["top_p"]
        p = torch.zeros_like(p).scatter(0, order, torch.where(keep, s, 0.0))
        p = p / p.sum()
    if c["min_p"] > 0.0:
        p = torch.where(p < p.max() * float(np.float32(c["min_p"])), 0.0, p)
        p = p / p.sum()
    return p

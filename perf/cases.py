"""What this library's users run, as measurable cases: the per-layer op set of an LLM (or speech encoder) forward
pass, called through ``sapient_amd.ops`` on device tensors.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call, ``run`` is one pass,
``exact`` the same results in 64 bits. The sizes are those of the repository's benchmark, tests and configurations
(Qwen2.5-0.5B, Llama-3-8B, phi-2 and Whisper shapes) and generic ones between them, odd ones included.

Kinds of case:
  layer    one decoder layer's share of the op set for `tokens` tokens: embedding gather, residual add + RMSNorm,
           bias + RoPE + KV-cache append, (chunks) the attention output's head transpose, residual add + RMSNorm, SwiGLU.
           The projections and attention between them are other libraries' work; their results are inputs here.
  encoder  a speech encoder's MLP block: LayerNorm, bias, erf-GELU, bias, residual add.
  norm     one norm over [rows, dim].
  act      one activation over [rows, dim].
  rope     rotary embedding of q and k, in place.
  embed    the embedding gather with GGUF row dequantization.
  kv       the KV-cache update of the trait path: append, sliding the window when the cache is full.
"""
import numpy as np
import torch

import sapient_amd.ops as ops
from sapient_amd._lib import BF16, F16, F32, Q4_K, Q8_0

DTYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
TABLE = {"f32": F32, "f16": F16, "bf16": BF16, "q8_0": Q8_0, "q4_k": Q4_K}
BLOCK = {"q8_0": (32, 34), "q4_k": (256, 144)}  # elements, bytes

# (hidden, heads, kv_heads, head_dim, intermediate, biases): decoder widths from 0.5 to 8 billion parameters
DECODERS = [(896, 14, 2, 64, 4864, True), (2048, 32, 8, 64, 8192, False), (2560, 32, 32, 80, 10240, True),
            (4096, 32, 8, 128, 14336, False)]


def listed():
    return [
        # One decode step of a 0.5B decoder (the benchmark's configuration 1, T = 1): the smallest calls, where
        # launches and call overhead are the time.
        dict(name="decode_step", kind="layer", tokens=1, hidden=896, heads=14, kv_heads=2, head_dim=64, inter=4864,
             biases=True, interleaved=False, dtype="f32", kv="f16", max_seq=4096, start=1000, table="q8_0",
             vocab=151936),
        # Its prefill in 512-token chunks (configuration 1, T = 512; the engine's chunk).
        dict(name="prefill_chunk", kind="layer", tokens=512, hidden=896, heads=14, kv_heads=2, head_dim=64,
             inter=4864, biases=True, interleaved=False, dtype="f32", kv="f16", max_seq=4096, start=512,
             table="q8_0", vocab=151936),
        # A whole prompt of odd length through an 8B decoder in bfloat16, GGUF rows (interleaved RoPE), Q4_K table.
        dict(name="prompt_8b_bf16", kind="layer", tokens=333, hidden=4096, heads=32, kv_heads=8, head_dim=128,
             inter=14336, biases=False, interleaved=True, dtype="bf16", kv="bf16", max_seq=8192, start=0,
             table="q4_k", vocab=128256),
        # The benchmark's headline: a large batch's fused residual add + RMSNorm in f32.
        dict(name="add_norm_f32", kind="norm", op="add_rms_norm", rows=16384, dim=4096, dtype="f32", w="f32",
             out="same"),
        # A width that no vector divides (pruned or probed models), ragged batch, half precision.
        dict(name="add_norm_ragged", kind="norm", op="add_rms_norm", rows=4099, dim=2565, dtype="f16", w="f32",
             out="same"),
        # 30 s of audio through a speech encoder's MLP block, half precision.
        dict(name="encoder_mlp", kind="encoder", rows=1500, dim=1280, inter=5120, dtype="f16"),
        # Long-prompt RoPE (configuration 3), half precision.
        dict(name="rope_8k_f16", kind="rope", batch=1, heads=32, kv_heads=8, seq=8192, head_dim=128, rotary=128,
             interleaved=False, start=0, dtype="f16"),
        # A large batch's gated activation (configuration 4): the largest activations.
        dict(name="swiglu_f16", kind="act", op="swiglu", rows=8192, dim=14336, dtype="f16", offset=0),
        # An odd-length prompt's GELU in the reference's own f32.
        dict(name="gelu_f32", kind="act", op="gelu_tanh", rows=777, dim=10240, dtype="f32", offset=0),
        # A large batch's gather from a 4-bit table (configuration 5).
        dict(name="embed_q4_k", kind="embed", table="q4_k", vocab=128256, hidden=4096, ids=65536, zipf=False),
        # A decode step on a full cache: the window slides by one row.
        dict(name="kv_slide_f16", kind="kv", n_kv=8, head_dim=128, max_seq=8192, cur_len=8192, seq=1, src="f32",
             cache="f16"),
        # A prefill chunk appended to a quantized cache.
        dict(name="kv_append_q8_0", kind="kv", n_kv=8, head_dim=128, max_seq=8192, cur_len=1000, seq=2048, src="f32",
             cache="q8_0"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "norm", "norm", "encoder", "rope", "act", "act", "embed", "kv", "kv"])
    dt = rng.choice(["f32", "f16", "bf16"])
    if kind == "layer":
        hidden, heads, kv_heads, head_dim, inter, biases = rng.choice(DECODERS)
        tokens = rng.choice([1, _log(rng, 2, 2048)])
        return dict(kind=kind, tokens=tokens, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                    inter=inter, biases=biases, interleaved=rng.random() < 0.3, dtype=dt,
                    kv=rng.choice(["f16", "bf16"] if dt == "f32" else [dt]), max_seq=4096,
                    start=rng.randrange(0, 4096 - tokens), table=rng.choice(["q8_0", "f16"] + ["q4_k"] * (hidden % 256 == 0)),
                    vocab=_log(rng, 32000, 151936))
    if kind == "encoder":
        dim = rng.choice([384, 512, 768, 1024, 1280])
        return dict(kind=kind, rows=_log(rng, 50, 12000), dim=dim, inter=4 * dim, dtype=dt)
    if kind == "norm":
        rows = _log(rng, 1, 16384)
        dim = rng.choice([64 * _log(rng, 2, 128), _log(rng, 100, 8192)])
        return dict(kind=kind, op=rng.choice(["add_rms_norm", "rms_norm", "layer_norm"]),
                    rows=min(rows, max(1, (1 << 26) // dim)), dim=dim, dtype=dt, w=rng.choice(["f32", "same"]),
                    out=rng.choice(["same", "same", "f32"]))
    if kind == "act":
        rows, dim = _log(rng, 1, 8192), rng.choice([128 * _log(rng, 3, 112), _log(rng, 300, 14336)])
        op = rng.choice(["swiglu", "gelu_tanh", "gelu_erf", "silu"])
        return dict(kind=kind, op=op, rows=min(rows, (1 << 26) // dim), dim=dim, dtype=dt,
                    offset=rng.choice([0, 0, 0, rng.randrange(1, 8)]))
    if kind == "rope":
        heads, kv_heads, head_dim, rotary = rng.choice([(14, 2, 64, 64), (32, 8, 128, 128), (32, 32, 80, 32),
                                                        (32, 8, 64, 64), (28, 4, 128, 128)])
        seq = _log(rng, 1, 8192)
        return dict(kind=kind, batch=rng.choice([1, 1, 3]) if seq < 2048 else 1, heads=heads, kv_heads=kv_heads,
                    seq=seq, head_dim=head_dim, rotary=rotary, interleaved=rng.random() < 0.4,
                    start=rng.randrange(0, 8193 - seq), dtype=dt)
    if kind == "embed":
        table = rng.choice(["q4_k", "q8_0", "f16", "bf16", "f32"])
        hidden = rng.choice([512, 896, 2048, 2560, 4096])
        return dict(kind=kind, table="q8_0" if table == "q4_k" and hidden % 256 else table,
                    vocab=_log(rng, 32000, 151936) if table != "f32" else 32000, hidden=hidden, ids=_log(rng, 1, 32768),
                    zipf=rng.random() < 0.5)
    n_kv, head_dim = rng.choice([(2, 64), (8, 128), (8, 64), (32, 80), (4, 128)])
    cache = rng.choice(["f16", "bf16", "q8_0", "q8_0"])
    if cache == "q8_0" and head_dim % 32:
        cache = "f16"
    max_seq = _log(rng, 512, 8192)
    seq = rng.choice([1, _log(rng, 2, max_seq)])
    cur = rng.choice([max_seq, rng.randrange(0, max_seq - seq + 1)])
    return dict(kind=kind, n_kv=n_kv, head_dim=head_dim, max_seq=max_seq, cur_len=cur, seq=seq,
                src=rng.choice(["f32", "f16"]), cache=cache)


# ───────────────────────────── inputs ─────────────────────────────
class _Make:
    """Seeded device tensors: activations ~N(0, std), one generator per case."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def randn(self, *shape, dtype=torch.float32, std=1.0, mean=0.0):
        return torch.randn(shape, generator=self.g, device=self.dev).mul_(std).add_(mean).to(dtype)

    def ids(self, n, vocab, zipf=False):
        if zipf:  # token frequencies of text, about 1 / rank
            r = torch.rand(n, generator=self.g, device=self.dev, dtype=torch.float64)
            return (float(vocab) ** r).long().clamp_(1, vocab).sub_(1).to(torch.int32)
        return torch.randint(0, vocab, (n,), generator=self.g, device=self.dev, dtype=torch.int32)

    def table(self, kind, vocab, hidden):
        """Raw GGUF table bytes (or a plain table)."""
        if kind in DTYPE:
            return self.randn(vocab, hidden, dtype=DTYPE[kind], std=0.02)
        elems, nbytes = BLOCK[kind]
        nb = vocab * hidden // elems
        t = torch.randint(0, 256, (nb, nbytes), generator=self.g, device=self.dev, dtype=torch.uint8)
        nd = 1 if kind == "q8_0" else 2
        d = torch.rand((nb, nd), generator=self.g, device=self.dev).mul_(0.02).add_(0.0005).to(torch.float16)
        t[:, :2 * nd] = d.view(torch.uint8).view(nb, 2 * nd)
        return t.view(-1)


def _offset(t, off):
    """The same values `off` elements into a larger allocation: a view that is only element-aligned."""
    if not off:
        return t
    raw = torch.empty(t.numel() + off, dtype=t.dtype, device=t.device)
    raw[off:].copy_(t.reshape(-1))
    return raw[off:].view(t.shape)


def prepare(case, seed):
    m, c, kind = _Make(seed), case, case["kind"]
    s = {"c": c}
    if kind == "layer":
        T, H, nq, nkv, D, dt = c["tokens"], c["hidden"], c["heads"], c["kv_heads"], c["head_dim"], DTYPE[c["dtype"]]
        s["table"] = m.table(c["table"], c["vocab"], H)
        s["ids"] = m.ids(T, c["vocab"])
        s["ln1"], s["ln2"] = m.randn(H, std=0.1, mean=1.0), m.randn(H, std=0.1, mean=1.0)
        s["down"], s["o"] = m.randn(T, H, dtype=dt), m.randn(T, H, dtype=dt)
        q, k, v = ((nq, T, D), (nkv, T, D), (nkv, T, D)) if T == 1 else ((T, nq, D), (T, nkv, D), (T, nkv, D))
        s["q"], s["k"], s["v"] = m.randn(*q, dtype=dt), m.randn(*k, dtype=dt), m.randn(*v, dtype=dt)
        s["b"] = [m.randn(n * D, std=0.1) for n in (nq, nkv, nkv)] if c["biases"] else [None] * 3
        s["pos"] = torch.arange(c["start"], c["start"] + T, dtype=torch.int32, device=m.dev)
        s["kc"], s["vc"] = (m.randn(nkv, c["max_seq"], D, dtype=DTYPE[c["kv"]]) for _ in range(2))
        s["attn"] = m.randn(nq, T, D, dtype=dt)
        s["gate"], s["up"] = m.randn(T, c["inter"], dtype=dt, std=2.0), m.randn(T, c["inter"], dtype=dt, std=2.0)
    elif kind == "encoder":
        dt, R, D = DTYPE[c["dtype"]], c["rows"], c["dim"]
        s["x"] = m.randn(R, D, dtype=dt, std=2.0, mean=0.3)
        s["w"], s["b"] = m.randn(D, std=0.1, mean=1.0), m.randn(D, std=0.1)
        s["fc1"], s["b1"] = m.randn(R, c["inter"], dtype=dt, std=1.5), m.randn(c["inter"], std=0.1)
        s["fc2"], s["b2"] = m.randn(R, D, dtype=dt), m.randn(D, std=0.1)
    elif kind == "norm":
        dt = DTYPE[c["dtype"]]
        wdt = dt if c["w"] == "same" else torch.float32
        s["x"] = m.randn(c["rows"], c["dim"], dtype=dt, mean=0.25 if c["op"] == "layer_norm" else 0.0)
        s["w"] = m.randn(c["dim"], dtype=wdt, std=0.1, mean=1.0)
        if c["op"] == "layer_norm":
            s["b"] = m.randn(c["dim"], dtype=wdt, std=0.1)
        if c["op"] == "add_rms_norm":
            s["r"] = m.randn(c["rows"], c["dim"], dtype=dt)
    elif kind == "act":
        shape, dt = (c["rows"], c["dim"]), DTYPE[c["dtype"]]
        s["x"] = _offset(m.randn(*shape, dtype=dt, std=2.0), c["offset"])
        if c["op"] == "swiglu":
            s["u"] = _offset(m.randn(*shape, dtype=dt, std=2.0), c["offset"])
        # Set-up that a program does once per process (the lookup tables of half-precision GELU).
        ops.init()
    elif kind == "rope":
        B, S, D, dt = c["batch"], c["seq"], c["head_dim"], DTYPE[c["dtype"]]
        s["q"], s["k"] = m.randn(B, c["heads"], S, D, dtype=dt), m.randn(B, c["kv_heads"], S, D, dtype=dt)
        s["pos"] = torch.arange(c["start"], c["start"] + S, dtype=torch.int32, device=m.dev)
    elif kind == "embed":
        s["table"] = m.table(c["table"], c["vocab"], c["hidden"])
        s["ids"] = m.ids(c["ids"], c["vocab"], c["zipf"])
    else:
        s["src"] = m.randn(c["n_kv"], c["seq"], c["head_dim"], dtype=DTYPE[c["src"]])
        if c["cache"] == "q8_0":
            nb = c["head_dim"] // 32
            t = torch.randint(0, 256, (c["n_kv"], c["max_seq"], nb, 34), generator=m.g, device=m.dev, dtype=torch.uint8)
            s["cache"] = t.view(c["n_kv"], c["max_seq"], nb * 34)
        else:
            s["cache"] = m.randn(c["n_kv"], c["max_seq"], c["head_dim"], dtype=DTYPE[c["cache"]])
    return s


THETA = {64: 1e6, 80: 1e4, 128: 5e5}
EPS = 1e-5


# ───────────────────────────── one pass ─────────────────────────────
def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "layer":
        x = ops.embed(s["table"], TABLE[c["table"]], c["vocab"], c["hidden"], s["ids"])
        if c["dtype"] != "f32":
            x = x.to(DTYPE[c["dtype"]])
        h, x = ops.add_rms_norm(s["down"], x, s["ln1"], EPS)
        bq, bk, bv = s["b"]
        base = THETA[c["head_dim"]]
        if c["tokens"] == 1:  # token-major and heads-major are the same layout; q is rotated in place
            ops.rope_kv_append(s["q"], s["k"], s["v"], s["pos"], base, s["kc"], s["vc"], interleaved=c["interleaved"],
                               bq=bq, bk=bk, bv=bv)
            q, att = s["q"], s["attn"]
        else:
            q = ops.rope_kv_append_tokens(s["q"], s["k"], s["v"], s["pos"], base, s["kc"], s["vc"],
                                          interleaved=c["interleaved"], bq=bq, bk=bk, bv=bv)
            att = ops.transpose_heads(s["attn"])
        h2, x = ops.add_rms_norm(s["o"], x, s["ln2"], EPS)
        act = ops.swiglu(s["gate"], s["up"])
        return {"h": h, "q": q, "kcache": s["kc"], "vcache": s["vc"], "attn": att, "x": x, "h2": h2, "act": act}
    if kind == "encoder":
        h = ops.layer_norm(s["x"], s["w"], s["b"], EPS)
        g = ops.gelu_erf(ops.add_bias(s["fc1"], s["b1"]))
        return {"h": h, "g": g, "x": ops.add(s["x"], ops.add_bias(s["fc2"], s["b2"]))}
    if kind == "norm":
        od = torch.float32 if c["out"] == "f32" else None
        if c["op"] == "add_rms_norm":
            return ops.add_rms_norm(s["x"], s["r"], s["w"], EPS, out_dtype=od)
        if c["op"] == "layer_norm":
            return ops.layer_norm(s["x"], s["w"], s["b"], EPS, out_dtype=od)
        return ops.rms_norm(s["x"], s["w"], EPS, out_dtype=od)
    if kind == "act":
        return ops.swiglu(s["x"], s["u"]) if c["op"] == "swiglu" else getattr(ops, c["op"])(s["x"])
    if kind == "rope":
        ops.rope_(s["q"], s["k"], s["pos"], THETA[c["head_dim"]], rotary_dim=c["rotary"], interleaved=c["interleaved"])
        return s["q"], s["k"]
    if kind == "embed":
        return ops.embed(s["table"], TABLE[c["table"]], c["vocab"], c["hidden"], s["ids"])
    n = ops.kv_cache_update(s["src"], s["cache"], c["cur_len"])
    return {"cache": s["cache"], "len": n}


# ───────────────────────────── bytes, operations, tolerances ─────────────────────────────
def _size(name):
    return 4 if name == "f32" else 2


def _row_bytes(table, hidden):
    return hidden * _size(table) if table in DTYPE else hidden // BLOCK[table][0] * BLOCK[table][1]


def work(case):
    c, kind = case, case["kind"]
    if kind == "layer":
        T, H, nq, nkv, D, e, kv = (c["tokens"], c["hidden"], c["heads"], c["kv_heads"], c["head_dim"], _size(c["dtype"]),
                                   _size(c["kv"]))
        b = T * (_row_bytes(c["table"], H) + 4)          # table rows and ids
        b += 6 * T * H * e + 8 * H                       # down, o in; h, h2, x out and x in again; norm weights
        b += 2 * T * nq * D * e + 2 * T * nkv * D * (e + kv) + 4 * T + c["biases"] * 4 * (nq + 2 * nkv) * D
        b += (T > 1) * 2 * T * nq * D * e                # the transpose
        b += 3 * T * c["inter"] * e
        return {"bytes": b, "flops": T * (12 * H + 4 * (nq + nkv) * D + 6 * c["inter"])}
    if kind == "encoder":
        e, n, ni = _size(c["dtype"]), c["rows"] * c["dim"], c["rows"] * c["inter"]
        return {"bytes": e * (4 * n + 2 * ni) + 4 * (3 * c["dim"] + c["inter"]), "flops": 10 * n + 20 * ni}
    if kind == "norm":
        e, n = _size(c["dtype"]), c["rows"] * c["dim"]
        o, w = (4 if c["out"] == "f32" else e), (4 if c["w"] == "f32" else e)
        add = c["op"] == "add_rms_norm"
        return {"bytes": n * (e * (3 if add else 1) + o) + c["dim"] * w * (2 if c["op"] == "layer_norm" else 1),
                "flops": n * (8 if c["op"] == "layer_norm" else 5)}
    if kind == "act":
        n = c["rows"] * c["dim"]
        return {"bytes": n * _size(c["dtype"]) * (3 if c["op"] == "swiglu" else 2),
                "flops": n * {"swiglu": 6, "silu": 5}.get(c["op"], 20)}
    if kind == "rope":
        n = c["batch"] * (c["heads"] + c["kv_heads"]) * c["seq"] * c["rotary"]
        return {"bytes": 2 * n * _size(c["dtype"]) + 4 * c["seq"], "flops": 3 * n}
    if kind == "embed":
        return {"bytes": c["ids"] * (_row_bytes(c["table"], c["hidden"]) + 4 + 4 * c["hidden"]),
                "flops": 2 * c["ids"] * c["hidden"]}
    shift = max(0, c["cur_len"] + c["seq"] - c["max_seq"])
    row = c["head_dim"] // 32 * 34 if c["cache"] == "q8_0" else c["head_dim"] * 2
    moved = 2 * (c["cur_len"] - shift) * row if shift else 0
    return {"bytes": c["n_kv"] * (moved + c["seq"] * (c["head_dim"] * _size(c["src"]) + row)),
            "flops": 4 * c["n_kv"] * c["seq"] * c["head_dim"] if c["cache"] == "q8_0" else 1}


def tolerance(case):
    c = case
    if c["kind"] in ("act", "rope", "embed", "kv"):
        return "exact"  # no sums: the library states these bit for bit
    # The norms' sums of squares: their order is free. Two orders measured (vector and element-wise kernels, up to
    # 16384 x 4096) differ by rel 6.7e-8 and max 4.7e-7 in f32; in 16 bits a few roundings turn to the neighbouring
    # value (rel 4.4e-6 in f16, 1.2e-5 in bf16, one unit in the last place at most). Four times the rel.
    if c["dtype"] == "f32":
        return {"rel": 3e-7, "max": 2e-6}
    return {"rel": 5e-5, "max": 0.008} if c["dtype"] == "bf16" else {"rel": 2e-5, "max": 0.001}


# ───────────────────────────── the same in 64 bits ─────────────────────────────
def _d(t):
    return None if t is None else t.double()


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * _d(w)


def _erf_as(x):
    """The Abramowitz-Stegun form that the reference defines erf-GELU by."""
    t = 1.0 / (1.0 + 0.3275911 * x.abs())
    p = ((((1.061405429 * t - 1.453152027) * t) + 1.421413741) * t - 0.284496736) * t + 0.254829592
    return torch.sign(x) * (1.0 - p * t * torch.exp(-x * x))


def _act(op, x, u=None):
    if op in ("swiglu", "silu"):
        y = x * torch.sigmoid(x)
        return y if u is None else y * u
    if op == "gelu_erf":
        return 0.5 * x * (1.0 + _erf_as(x * 0.5 ** 0.5))
    return 0.5 * x * (1.0 + torch.tanh(0.79788456 * (x + 0.044715 * x ** 3)))


def _rope(x, pos, base, rotary, interleaved):
    """x [..., tokens, head_dim] in f64; the angle itself is f32 by the reference's definition."""
    den = np.power(np.float32(base), np.arange(0, rotary, 2, dtype=np.float32) / np.float32(rotary), dtype=np.float32)
    ang = (pos.float()[:, None] / torch.from_numpy(den).to(x.device)).double()
    cs, sn = ang.cos(), ang.sin()
    y = x.clone()
    a = slice(0, rotary, 2) if interleaved else slice(0, rotary // 2)
    b = slice(1, rotary, 2) if interleaved else slice(rotary // 2, rotary)
    y[..., a] = x[..., a] * cs - x[..., b] * sn
    y[..., b] = x[..., b] * cs + x[..., a] * sn
    return y


def _embed(s, c):
    ids, H = s["ids"].long(), c["hidden"]
    if c["table"] in DTYPE:
        return s["table"][ids].double()
    elems, nbytes = BLOCK[c["table"]]
    r = s["table"].view(c["vocab"], H // elems, nbytes)[ids]
    if c["table"] == "q8_0":
        d = r[..., :2].contiguous().view(torch.float16).double()
        return (r[..., 2:].contiguous().view(torch.int8).double() * d).reshape(-1, H)
    d = r[..., 0:2].contiguous().view(torch.float16).double()
    dmin = r[..., 2:4].contiguous().view(torch.float16).double()
    sb = r[..., 4:16].int()
    lo, mid, hi = sb[..., 0:4], sb[..., 4:8], sb[..., 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double()
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1).double()
    q = r[..., 16:].view(*r.shape[:2], 4, 32).int()
    q = torch.stack([q & 15, q >> 4], -2).reshape(*r.shape[:2], 8, 32).double()
    return (d[..., None] * sc[..., None] * q - dmin[..., None] * mn[..., None]).reshape(-1, H)


def exact(case, seed):
    s, c, kind = prepare(case, seed), case, case["kind"]
    if kind == "layer":
        x = _embed(s, c)
        x = x + _d(s["down"])
        h = _rms(x, s["ln1"])
        T, nq, nkv, D = c["tokens"], c["heads"], c["kv_heads"], c["head_dim"]
        q, k, v = _d(s["q"]), _d(s["k"]), _d(s["v"])
        if T > 1:
            q, k, v = (t.transpose(0, 1) for t in (q, k, v))
        bq, bk, bv = (0.0 if b is None else _d(b).view(-1, 1, D) for b in s["b"])
        q, k = (_rope(t, s["pos"], THETA[D], D, c["interleaved"]) for t in (q + bq, k + bk))
        kc, vc = _d(s["kc"]), _d(s["vc"])
        kc[:, c["start"]:c["start"] + T], vc[:, c["start"]:c["start"] + T] = k, v + bv
        att = _d(s["attn"]) if T == 1 else _d(s["attn"]).transpose(0, 1).contiguous()
        x = x + _d(s["o"])
        return {"h": h, "q": q.contiguous(), "kcache": kc, "vcache": vc, "attn": att, "x": x, "h2": _rms(x, s["ln2"]),
                "act": _act("swiglu", _d(s["gate"]), _d(s["up"]))}
    if kind == "encoder":
        h = torch.nn.functional.layer_norm(_d(s["x"]), (c["dim"],), _d(s["w"]), _d(s["b"]), EPS)
        # The activation reads the sum as its type holds it.
        y = (s["fc1"].float() + s["b1"]).to(s["fc1"].dtype).double()
        return {"h": h, "g": _act("gelu_erf", y), "x": _d(s["x"]) + _d(s["fc2"]) + _d(s["b2"])}
    if kind == "norm":
        x = _d(s["x"])
        if c["op"] == "layer_norm":
            return torch.nn.functional.layer_norm(x, (c["dim"],), _d(s["w"]), _d(s["b"]), EPS)
        if c["op"] == "rms_norm":
            return _rms(x, s["w"])
        r = x + _d(s["r"])
        return _rms(r, s["w"]), r
    if kind == "act":
        return _act(c["op"], _d(s["x"]), _d(s["u"]) if c["op"] == "swiglu" else None)
    if kind == "rope":
        return tuple(_rope(_d(s[n]), s["pos"], THETA[c["head_dim"]], c["rotary"], c["interleaved"]) for n in "qk")
    if kind == "embed":
        return _embed(s, c)
    n = min(c["cur_len"] + c["seq"], c["max_seq"])
    if c["cache"] == "q8_0":
        return {"cache": None, "len": n}  # quantized bytes
    y, shift = _d(s["cache"]), c["cur_len"] + c["seq"] - n
    y[:, :n - c["seq"]] = y[:, shift:c["cur_len"]].clone()
    y[:, n - c["seq"]:n] = _d(s["src"])
    return {"cache": y, "len": n}

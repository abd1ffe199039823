"""Performance cases of the Q4/g64 decoder path, each one a call sequence that a program
using this library makes, over the sizes of the Gemma-class 12B decoder (synthetic.py:
hidden 3840, intermediate 15360, 16 query heads, sliding layers of 8 KV heads x 256 with a
1024-token window, global layers of 1 KV head x 512 with K = V, vocabulary 262144).

Kinds:
  proj      one quantized projection of m rows (hyp_qmatmul)
  mlp       the feed-forward block: fused gate/up + GELU, then down
  attn      the attention block after the residual stream: input norm + q/k/v, the per-head
            norms with RoPE and the cache append, attention over the cache, o
  sample    the temperature draw with its top-8 sidecar over one row of logits
  quantize  quantize/pack of a bf16 matrix
  model     one request through the model-level entry points: a new KV state, the prompt's
            prefill, a block of greedy decode steps with the top-8 logits, the state freed

Weights and activations are random (seeded), made on the GPU with torch; the exact()
results are float64 torch on the same inputs.
"""
import ctypes
import math
import os
import shutil
import tempfile

import numpy as np
import torch

import hyperion_amd as hy
from hyperion_amd import synthetic as syn

EPS = 1e-6
HEADS = 16
WINDOW = 1024
RING = WINDOW + 2048          # a sliding layer's cache, as the decoder sizes it
SHAPES = ((15360, 3840), (3840, 15360), (4096, 3840), (8192, 3840), (2048, 3840), (3840, 4096), (3840, 8192))

_stream = None
_model = None


def stream():
    """The one stream of this program."""
    global _stream
    if _stream is None:
        _stream = hy.Stream()
    return _stream


class Buf(hy.DeviceArray):
    """A torch tensor's memory as the device array that the entry points take."""

    def __init__(self, tensor):
        self.tensor = tensor
        self._p = ctypes.c_void_p(tensor.data_ptr())

    def close(self):
        pass


class _Raw:
    """Library memory (a cache's rows) for torch.as_tensor; the tensor keeps this object, and
    with it the owner of the memory, alive."""

    def __init__(self, owner, address, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (address, False), "shape": tuple(shape), "typestr": "<i2",
                                         "version": 2}


def listed():
    return [
        # The decode GEMV of the benchmark (gate or up of one token): the smallest call.
        {"name": "gemv", "kind": "proj", "n": 15360, "k": 3840, "m": 1},
        # Four sequences decoded together, the largest batch of the decode kernel's range.
        {"name": "mlp-4", "kind": "mlp", "m": 4},
        # Sixteen sequences decoded together, or a 16-token prompt.
        {"name": "mlp-16", "kind": "mlp", "m": 16},
        # A short prompt of an odd length.
        {"name": "mlp-203", "kind": "mlp", "m": 203},
        # A whole prefill chunk.
        {"name": "mlp-2048", "kind": "mlp", "m": 2048},
        # One decode step of a sliding layer with a full window behind it.
        {"name": "attn-decode-sliding", "kind": "attn", "layer": "sliding", "m": 1, "offset": 1500},
        # One decode step of a global layer in a long conversation.
        {"name": "attn-decode-global", "kind": "attn", "layer": "global", "m": 1, "offset": 30001},
        # A prompt of ordinary length behind an earlier turn, sliding layer.
        {"name": "attn-prefill-sliding", "kind": "attn", "layer": "sliding", "m": 1000, "offset": 700},
        # The second whole chunk of a long prompt, global layer.
        {"name": "attn-prefill-global", "kind": "attn", "layer": "global", "m": 2048, "offset": 2048},
        # One sampled token at the model's vocabulary.
        {"name": "sample", "kind": "sample", "vocab": 262144, "temperature": 0.8, "top_k": 64, "top_p": 0.95,
         "min_p": 0.05},
        # Quantizing the gate projection.
        {"name": "quantize", "kind": "quantize", "n": 15360, "k": 3840},
        # A request to a six-layer model of the 12B's layer and vocabulary sizes.
        {"name": "request", "kind": "model", "prompt": 1111, "decode": 32},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("proj", "proj", "mlp", "mlp", "attn", "attn", "attn", "sample", "quantize", "model"))
    if kind == "proj":
        n, k = rng.choice(SHAPES)
        return {"kind": kind, "n": n, "k": k, "m": _log(rng, 1, 2048)}
    if kind == "mlp":
        return {"kind": kind, "m": _log(rng, 1, 2047)}
    if kind == "attn":
        layer = rng.choice(("sliding", "global"))
        if rng.random() < 0.5:   # a decode step
            return {"kind": kind, "layer": layer, "m": 1, "offset": _log(rng, 16, 60000 if layer == "global" else 20000)}
        m = _log(rng, 2, 2047)
        return {"kind": kind, "layer": layer, "m": m, "offset": rng.choice((0, _log(rng, 5, 4095 - m)))}
    if kind == "sample":
        return {"kind": kind, "vocab": _log(rng, 1000, 262143), "temperature": round(rng.uniform(0.3, 1.5), 2),
                "top_k": rng.choice((0, 20, 64)), "top_p": rng.choice((0.9, 0.95, 1.0)),
                "min_p": rng.choice((0.0, 0.05))}
    if kind == "quantize":
        k = 64 * _log(rng, 4, 240)
        return {"kind": kind, "n": min(_log(rng, 16, 15359), 15360 * 3840 // k), "k": k}
    return {"kind": kind, "prompt": _log(rng, 2, 1100), "decode": rng.randint(4, 32)}


# ---- inputs -----------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _q4(g, n, k):
    """Codes, scales and biases (MLX layout) of a projection whose rows have unit gain."""
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    u = torch.rand((n, k // 64), generator=g, device="cuda") + 0.5
    s = (u / (4.61 * math.sqrt(k))).to(torch.bfloat16)
    return w, s, (s.float() * -7.5).to(torch.bfloat16)


def _norm(g, n, around=1.0):
    return (around * (1.0 + 0.1 * _randn(g, n))).to(torch.bfloat16)


def _attn_sizes(case):
    sliding = case["layer"] == "sliding"
    d, kvh = (256, 8) if sliding else (512, 1)
    m, offset = case["m"], case["offset"]
    if sliding and offset % RING + m > RING:   # the chunk's slots in one piece
        offset -= offset % RING + m - RING
    prefix = min(WINDOW, offset) if sliding else offset
    cap = RING if sliding else offset + m
    return sliding, d, kvh, m, offset, prefix, cap


def _inputs(case, seed):
    """The random tensors of a case, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    t = {}
    if kind == "proj":
        t["w"] = _q4(g, case["n"], case["k"])
        t["x"] = _randn(g, case["m"], case["k"]).to(torch.bfloat16)
    elif kind == "mlp":
        t["gate"], t["up"], t["down"] = _q4(g, 15360, 3840), _q4(g, 15360, 3840), _q4(g, 3840, 15360)
        t["x"] = _randn(g, case["m"], 3840).to(torch.bfloat16)
    elif kind == "attn":
        sliding, d, kvh, m, _, prefix, _ = _attn_sizes(case)
        t["q"], t["k"] = _q4(g, HEADS * d, 3840), _q4(g, kvh * d, 3840)
        if sliding:
            t["v"] = _q4(g, kvh * d, 3840)
        t["o"] = _q4(g, 3840, HEADS * d)
        t["x"] = _randn(g, m, 3840).to(torch.bfloat16)
        t["norm"] = _norm(g, 3840)
        t["q_norm"], t["k_norm"] = _norm(g, d, d ** -0.25), _norm(g, d, d ** -0.25)
        t["pk"] = (d ** -0.25 * _randn(g, prefix, kvh, d)).to(torch.bfloat16)
        t["pv"] = _randn(g, prefix, kvh, d).to(torch.bfloat16)
    elif kind == "sample":
        t["logits"] = (30.0 * torch.tanh(3.0 * _randn(g, case["vocab"]) / 30.0)).to(torch.bfloat16)
    elif kind == "quantize":
        w = (0.02 * _randn(g, case["n"], case["k"])).to(torch.bfloat16)
        big = torch.rand(w.shape, generator=g, device="cuda") < 0.01
        t["w"] = torch.where(big, w * 8, w)
    elif kind == "model":
        t["tokens"] = torch.randint(0, syn.VOCAB, (case["prompt"],), generator=g, device="cuda")
    return t


def _qweight(parts):
    w, s, b = parts
    n, k = w.shape[0], s.shape[1] * 64
    h = ctypes.c_void_p()
    hy.call("hyp_qweight_create_device", w.data_ptr(), s.data_ptr(), b.data_ptr(), n, k, 64, 4, stream().handle,
            ctypes.byref(h))
    return hy.QWeight(h)


def _empty(*shape, dtype=torch.bfloat16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _the_model():
    """The served model: loaded once, as a serving program does. Small branch gains keep every
    greedy choice far from a tie (the head is the embedding), so the tokens fed back do not
    hang on the rounding of one layer."""
    global _model
    if _model is None:
        cfg = syn.gemma4_text_config(num_layers=6)
        d = tempfile.mkdtemp(prefix="hyp_cases_")
        try:
            syn.write_model(d, cfg, seed=11, branch_gain=0.1, share_layers=True)
            _model = hy.Model(hy.geometry_from_config(cfg), os.path.join(d))
        finally:
            shutil.rmtree(d, ignore_errors=True)
    return _model


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    torch.cuda.synchronize()   # torch fills the inputs on its own stream
    if kind == "proj":
        st["w"], st["x"] = _qweight(t["w"]), Buf(t["x"])
        st["y"] = Buf(_empty(case["m"], case["n"]))
    elif kind == "mlp":
        for name in ("gate", "up", "down"):
            st[name] = _qweight(t[name])
        st["x"], st["h"], st["y"] = Buf(t["x"]), Buf(_empty(case["m"], 15360)), Buf(_empty(case["m"], 3840))
    elif kind == "attn":
        sliding, d, kvh, m, offset, prefix, cap = _attn_sizes(case)
        names = ("q", "k", "v") if sliding else ("q", "k")
        st["qkv"] = [_qweight(t[n]) for n in names]
        st["qkv_out"] = [Buf(_empty(m, (HEADS if n == "q" else kvh) * d)) for n in names]
        st["o"] = _qweight(t["o"])
        for name in ("x", "norm", "q_norm", "k_norm"):
            st[name] = Buf(t[name])
        st["attn"], st["y"] = Buf(_empty(m, HEADS * d)), Buf(_empty(m, 3840))
        st["cache"] = cache = hy.KvCache(cap, kvh, d)
        if prefix:
            pk, pv = Buf(t["pk"]), Buf(t["pv"])
            cache.write(pk, pv, prefix, offset - prefix, stream())
        ck, cv = cache.buffers()
        row = 2 * kvh * d * (offset % cap)
        st["new"] = [torch.as_tensor(_Raw(cache, p.value + row, (m, kvh * d)), device="cuda").view(torch.bfloat16)
                     for p in (ck, cv)]
        st["at"] = (sliding, d, m, offset, prefix)
    elif kind == "sample":
        st["logits"], st["out"] = Buf(t["logits"]), Buf(_empty(20, dtype=torch.int32))
        st["cfg"] = hy.SamplingConfig(case["temperature"], case["top_k"], case["top_p"], case["min_p"], seed)
        st["rng"] = seed * 2654435761 + 12345
    elif kind == "quantize":
        n, k = case["n"], case["k"]
        st["w"], st["codes"] = Buf(t["w"]), Buf(_empty(n, k // 8, dtype=torch.int32))
        st["s"], st["b"] = Buf(_empty(n, k // 64)), Buf(_empty(n, k // 64))
    elif kind == "model":
        st["model"] = _the_model()
        st["tokens"] = t["tokens"].cpu().numpy().astype(np.uint32)
        st["result"] = hy.StepResult()
    stream().synchronize()     # the uploads read the tensors made above
    torch.cuda.synchronize()
    return st


# ---- one pass ---------------------------------------------------------------------------

def _fields(f):
    return {"token": int(f.token_id), "logit": float(f.logit),
            "top": np.array(f.top_k_logprob_values[:f.top_k_logprob_count], np.float32)}


def run(st):
    s = stream()
    case, kind = st["case"], st["kind"]
    if kind == "proj":
        hy.qmatmul(st["w"], st["x"], case["m"], st["y"], s)
        return st["y"].tensor
    if kind == "mlp":
        hy.qmlp_gate_up_gelu(st["gate"], st["up"], st["x"], case["m"], st["h"], s)
        hy.qmatmul(st["down"], st["h"], case["m"], st["y"], s)
        return {"h": st["h"].tensor, "y": st["y"].tensor}
    if kind == "attn":
        sliding, d, m, offset, prefix = st["at"]
        q, k = st["qkv_out"][:2]
        v = st["qkv_out"][2] if sliding else None
        hy.qmatmul_group(st["qkv"], st["x"], m, st["qkv_out"], s, rms_eps=EPS, norm_weight=st["norm"])
        hy.attention_prepare(q, k, v, m, HEADS, st["cache"], st["q_norm"], st["k_norm"], EPS,
                             256 if sliding else 128, 1e4 if sliding else 1e6, offset, s)
        hy.call("hyp_attention", q.ptr, None, None, m, HEADS, st["cache"].handle, offset, prefix,
                WINDOW if sliding else 0, st["attn"].ptr, s.handle)
        hy.qmatmul(st["o"], st["attn"], m, st["y"], s)
        return {"k": st["new"][0], "v": st["new"][1], "attn": st["attn"].tensor, "y": st["y"].tensor}
    if kind == "sample":
        hy.sample_stochastic(st["logits"], case["vocab"], st["cfg"], st["rng"], st["out"], s)
        return st["out"].tensor
    if kind == "quantize":
        hy.quantize(st["w"], case["n"], case["k"], st["codes"], st["s"], st["b"], s)
        return {"codes": st["codes"].tensor, "s": st["s"].tensor, "b": st["b"].tensor}
    kv = st["model"].kvstate()
    try:
        first = _fields(kv.prefill(st["tokens"], st["result"], sampled=True))
        last = _fields(kv.decode(case["decode"], st["result"], sampled=True))
    finally:
        kv.close()
    return {"first": first, "last": last}


# ---- what a pass has to do, and how exactly ---------------------------------------------

def _q4_bytes(n, k):
    return n * k // 2 + 4 * n * (k // 64)


def _attn_pairs(m, prefix, window):
    """Visible (query, key) pairs of a chunk of m behind a prefix."""
    total = 0
    for t in range(m):
        seen = prefix + t + 1
        total += min(seen, window) if window else seen
    return total


def work(case):
    kind = case["kind"]
    if kind == "proj":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": _q4_bytes(n, k) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "mlp":
        m = case["m"]
        return {"bytes": 2 * _q4_bytes(15360, 3840) + _q4_bytes(3840, 15360) + 2 * m * (2 * 3840 + 2 * 15360),
                "flops": 6 * m * 3840 * 15360}
    if kind == "attn":
        sliding, d, kvh, m, offset, prefix, _ = _attn_sizes(case)
        shapes = [(HEADS * d, 3840), (kvh * d, 3840), (3840, HEADS * d)] + ([(kvh * d, 3840)] if sliding else [])
        w = WINDOW if sliding else 0
        weights = sum(_q4_bytes(n, k) for n, k in shapes)
        cached = min(prefix, WINDOW - 1) if sliding else prefix   # the oldest key a window still shows
        act = 2 * m * (2 * 3840 + 2 * kvh * d + 2 * HEADS * d) + 4 * kvh * d * cached
        flops = 2 * m * sum(n * k for n, k in shapes) + 4 * HEADS * d * _attn_pairs(m, prefix, w)
        return {"bytes": weights + act, "flops": flops}
    if kind == "sample":
        return {"bytes": 2 * case["vocab"] + 80, "flops": 0}
    if kind == "quantize":
        nk = case["n"] * case["k"]
        return {"bytes": 2 * nk + nk // 2 + 4 * nk // 64, "flops": 0}
    p, dec = case["prompt"], case["decode"]
    sl = sum(_q4_bytes(n, k) for n, k in syn.LAYER_SHAPES.values())
    gl = sum(_q4_bytes(n, k) for n, k in ((8192, 3840), (512, 3840), (3840, 8192), (15360, 3840), (15360, 3840),
                                          (3840, 15360)))
    weights, head = 5 * sl + gl, _q4_bytes(syn.VOCAB, 3840)
    params = 2 * (5 * sum(n * k for n, k in syn.LAYER_SHAPES.values()) + 16 * 3840 * 512 * 2 + 512 * 3840 +
                  3 * 15360 * 3840)
    keys = 5 * 8 * 256 * min(p, WINDOW) + 512 * p
    attn = 4 * HEADS * (5 * 256 * _attn_pairs(p, 0, WINDOW) + 512 * _attn_pairs(p, 0, 0))
    return {"bytes": (1 + dec) * (weights + head) + dec * 4 * keys, "flops": p * params + attn}


def tolerance(case):
    """About four times the bf16 rounding seen against exact(): 2e-3 for one projection, 5e-3
    for the feed-forward block, 6.5e-3 for the attention block."""
    kind = case["kind"]
    if kind in ("sample", "quantize"):
        return "exact"
    if kind == "proj":
        return {"rel": 1e-2}
    if kind == "mlp":
        return {"rel": 2e-2}
    if kind == "attn":
        return {"rel": 2.5e-2}
    return {"rel": 2e-2}


# ---- the same in float64 ------------------------------------------------------------------

def _dense(parts):
    """Dequantized weights, exactly scale * q + bias."""
    w, s, b = parts
    shifts = torch.arange(0, 32, 4, device=w.device, dtype=torch.int64)
    q = ((w.to(torch.int64)[:, :, None] >> shifts) & 15).reshape(w.shape[0], -1).to(torch.float64)
    g = s.shape[1]
    q = q.reshape(q.shape[0], g, 64) * s.double()[:, :, None] + b.double()[:, :, None]
    return q.reshape(q.shape[0], g * 64)


def _apply(x, parts):
    return x @ _dense(parts).t()


def _rms(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _rope(x, rotated, base, offset):
    """x [m, heads, d]; angles are float32 products, as the reference forms them."""
    m, _, d = x.shape
    half = d // 2
    inv = (base ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / d)).float()
    pos = torch.arange(offset, offset + m, device=x.device).float()
    theta = (pos[:, None] * inv[None, :]).double()
    theta[:, rotated // 2:] = 0.0
    c, s = torch.cos(theta)[:, None, :], torch.sin(theta)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, a * s + b * c), dim=-1)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("proj", "mlp", "attn"):
        return None
    t = _inputs(case, seed)
    x = t["x"].double()
    if kind == "proj":
        return _apply(x, t["w"])
    if kind == "mlp":
        h = _gelu(_apply(x, t["gate"])) * _apply(x, t["up"])
        return {"h": h, "y": _apply(h, t["down"])}
    sliding, d, kvh, m, offset, prefix, _ = _attn_sizes(case)
    xn = _rms(x, t["norm"])
    rot, base = (256, 1e4) if sliding else (128, 1e6)
    q = _rope(_rms(_apply(xn, t["q"]).reshape(m, HEADS, d), t["q_norm"]), rot, base, offset)
    raw = _apply(xn, t["k"]).reshape(m, kvh, d)
    k = _rope(_rms(raw, t["k_norm"]), rot, base, offset)
    v = _rms(_apply(xn, t["v"]).reshape(m, kvh, d) if sliding else raw)
    keys, vals = torch.cat((t["pk"].double(), k)), torch.cat((t["pv"].double(), v))
    qi = prefix + torch.arange(m, device=x.device)[:, None]
    kj = torch.arange(prefix + m, device=x.device)[None, :]
    seen = kj <= qi
    if sliding:
        seen &= kj > qi - WINDOW
    out = torch.empty((m, HEADS, d), dtype=torch.float64, device=x.device)
    for h in range(HEADS):
        j = h // (HEADS // kvh)
        sc = q[:, h].contiguous() @ keys[:, j].t().contiguous()
        out[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), dim=-1) @ vals[:, j].contiguous()
    out = out.reshape(m, HEADS * d)
    return {"k": k.reshape(m, kvh * d), "v": v.reshape(m, kvh * d), "attn": out, "y": _apply(out, t["o"])}

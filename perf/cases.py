"""What the performance of this library is measured on: calls that a program which runs a Llama- or Qwen-style model
over HipBackend makes, each through the Python binding's public entry points.

A case is one pass of one kind of work:
  attn   append_rope_attention / append_rope_attention_f16kv of one layer: a decode step (n = 1), a short append, a
         prompt chunk on a filled cache, or a whole prompt
  batch  append_rope_attention_batch of one layer: many sequences of different lengths, one token each
  proj   the layer's Q, K and V projections: matmul_multi (and add_bias where the model has biases)
  mlp    the layer's feed-forward block: rmsnorm, gate and up, silu_mul, down, residual add
  head   the last norm and the vocabulary projection: the logits of the last token of n sequences
  model  a whole forward of a few layers: embed to logits, as a program's decode step or prompt chunk runs it

Head shapes are those of nibble_amd.configs and generic ones; widths are those of the configurations and the
benchmark (896, 2048, 8192) and generic ones. Weight types are the float one that models ship in (F16) and the block
formats of common model files (Q4_0, Q5_0, Q8_0; Q4_K with Q6_K for the down projection and the head; Q5_K).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import nibble_amd
from nibble_amd import synth

EPS = 1e-5
DEV = "cuda"

# weight type: ggml id, elements per block, bytes per block
TYPES = {"f32": (nibble_amd.F32, 1, 4), "f16": (nibble_amd.F16, 1, 2), "q4_0": (nibble_amd.Q4_0, 32, 18),
         "q5_0": (nibble_amd.Q5_0, 32, 22), "q8_0": (nibble_amd.Q8_0, 32, 34), "q4_k": (nibble_amd.Q4_K, 256, 144),
         "q5_k": (nibble_amd.Q5_K, 256, 176), "q6_k": (nibble_amd.Q6_K, 256, 210)}


def listed():
    return [
        # one layer of a decode step early in a chat with a small model: latency, launches
        dict(name="decode_short", kind="attn", heads=14, kv_heads=2, head_dim=64, neox=True, base=1e6, llama3=False,
             n=1, pos0=512, cache="f32"),
        # the benchmark's decode step: a 32k context, HBM
        dict(name="decode_32k", kind="attn", heads=32, kv_heads=8, head_dim=64, neox=False, base=5e5, llama3=True,
             n=1, pos0=32768, cache="f32"),
        # a decode step over the opt-in fp16 cache at a middling, odd context and the larger head size
        dict(name="decode_f16kv", kind="attn", heads=32, kv_heads=8, head_dim=128, neox=False, base=5e5, llama3=True,
             n=1, pos0=6001, cache="f16"),
        # serving: 16 sequences of 1k..128k tokens (the benchmark's ragged step)
        dict(name="decode_ragged_16", kind="batch", heads=32, kv_heads=8, head_dim=64, neox=False, base=5e5,
             llama3=True, n_seq=16, lo=1024, hi=131072, lengths_seed=5),
        # a long prompt in one call (the benchmark's prefill)
        dict(name="prefill_8k", kind="attn", heads=32, kv_heads=8, head_dim=64, neox=False, base=5e5, llama3=True,
             n=8192, pos0=0, cache="f32"),
        # a later chunk of a prompt, ragged
        dict(name="prefill_chunk", kind="attn", heads=32, kv_heads=4, head_dim=64, neox=False, base=1e4, llama3=False,
             n=509, pos0=3072, cache="f32"),
        # projections of a prompt chunk, F16 weights
        dict(name="qkv_f16_chunk", kind="proj", width=2048, q_rows=2048, kv_rows=512, wtype="f16", bias=False, n=512),
        # feed-forward of a prompt chunk, the common 4-bit mix
        dict(name="mlp_q4k_chunk", kind="mlp", width=2048, ff=8192, wtype="q4_k", down_type="q6_k", n=512),
        # feed-forward of a short ragged prompt of a small 8-bit model
        dict(name="mlp_q8_0_short", kind="mlp", width=896, ff=3584, wtype="q8_0", down_type="q8_0", n=77),
        # feed-forward of a decode step, the common 4-bit mix
        dict(name="mlp_q4k_decode", kind="mlp", width=2048, ff=8192, wtype="q4_k", down_type="q6_k", n=1),
        # logits of one token over a large vocabulary
        dict(name="head_q6k", kind="head", width=2048, vocab=131072, wtype="q6_k", n=1),
        # a whole decode step of a small stack, embed to logits
        dict(name="model_decode", kind="model", layers=4, heads=32, kv_heads=8, head_dim=64, neox=False, base=5e5,
             llama3=True, ff=8192, vocab=32768, wtype="q4_k", down_type="q6_k", n=1, pos0=1500),
    ]


# ---- drawn cases ----

HEADS = [(14, 2, 64, True, 1e6, False), (32, 4, 64, False, 1e4, False), (32, 8, 64, False, 5e5, True),
         (32, 8, 128, False, 5e5, True), (24, 8, 128, False, 5e5, True), (12, 12, 64, True, 1e6, False)]
MAX_FLOPS = 2.7e11  # of the largest listed case
MAX_BYTES = 1.8e9


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _heads(rng):
    h, kv, hd, neox, base, l3 = rng.choice(HEADS)
    return dict(heads=h, kv_heads=kv, head_dim=hd, neox=neox, base=base, llama3=l3)


def _rows(rng):
    return 1 if rng.random() < 0.35 else _log_int(rng, 2, 640)


def _wtypes(rng, width):
    w = rng.choice(["f16", "f16", "q8_0", "q4_0", "q5_0"] +
                   (["q4_k", "q4_k", "q4_k", "q5_k", "q6_k"] if width % 256 == 0 else []))
    return w, "q6_k" if w in ("q4_k", "q5_k") else w


def _width(rng, lo, hi):
    """Widths as models have them: a multiple of 128 (K formats apply only to multiples of 256)."""
    return max(lo, _log_int(rng, lo, hi) // 128 * 128)


def _draw(rng):
    kind = rng.choice(["attn"] * 4 + ["batch", "proj", "proj", "mlp", "mlp", "mlp", "head", "model"])
    if kind == "attn":
        c = dict(kind=kind, **_heads(rng), cache=rng.choice(["f32", "f32", "f16"]))
        what = rng.random()
        if what < 0.45:
            c.update(n=1, pos0=_log_int(rng, 16, 65536))
        elif what < 0.55:
            c.update(n=_log_int(rng, 2, 16), pos0=_log_int(rng, 16, 16384))
        elif what < 0.8:
            c.update(n=_log_int(rng, 17, 1024), pos0=_log_int(rng, 1, 16384))
        else:
            c.update(n=_log_int(rng, 17, 8192), pos0=0)
        return c
    if kind == "batch":
        return dict(kind=kind, **_heads(rng), n_seq=_log_int(rng, 2, 31), lo=rng.choice([64, 1024]),
                    hi=_log_int(rng, 2048, 65536), lengths_seed=rng.randrange(1 << 20))
    width = _width(rng, 512, 3072)
    wtype, down = _wtypes(rng, width)
    if kind == "proj":
        kv = rng.choice([128, 256, 512, 1024])
        return dict(kind=kind, width=width, q_rows=width, kv_rows=kv, wtype=wtype, bias=rng.random() < 0.3,
                    n=_rows(rng))
    if kind == "mlp":
        ff = _width(rng, 1024, 8192)
        if TYPES[down][1] == 256:
            ff = ff // 256 * 256
        return dict(kind=kind, width=width, ff=ff, wtype=wtype, down_type=down, n=_rows(rng))
    if kind == "head":
        return dict(kind=kind, width=width, vocab=_log_int(rng, 16000, 110000), wtype=down,
                    n=rng.choice([1, 1, 1, 2, 5, 16]))
    h = dict(rng.choice([dict(heads=32, kv_heads=8, head_dim=64, neox=False, base=5e5, llama3=True, ff=8192),
                         dict(heads=14, kv_heads=2, head_dim=64, neox=True, base=1e6, llama3=False, ff=3584)]))
    wtype, down = _wtypes(rng, h["heads"] * h["head_dim"])
    return dict(kind=kind, layers=rng.choice([2, 3, 4]), **h, vocab=32768, wtype=wtype, down_type=down,
                n=1 if rng.random() < 0.6 else _log_int(rng, 2, 512), pos0=_log_int(rng, 1, 4096))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return c


# ---- work: each input read once, each output written once ----

def _wbytes(wtype, rows, width):
    _, be, bb = TYPES[wtype]
    return rows * width // be * bb


def _lengths(case):
    """The batch's cache lengths: log-uniform in [lo, hi]."""
    u = np.random.default_rng(case["lengths_seed"]).random(case["n_seq"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [int(round(math.exp(lo + (hi - lo) * x))) for x in u]


def _attn_work(h, kv, hd, n, pos0, elem):
    keys = n * pos0 + n * (n + 1) // 2
    return (2 * n * h * hd * 4 + 2 * pos0 * kv * hd * elem + 2 * n * kv * hd * (4 + elem)), 4 * h * hd * keys


def _matmul_work(wtype, rows, width, n):
    return _wbytes(wtype, rows, width) + 4 * n * (width + rows), 2 * n * rows * width


def _add(*parts):
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def _mlp_work(c, width):
    n, ff = c["n"], c["ff"]
    w = _wbytes(c["wtype"], 2 * ff, width) + _wbytes(c["down_type"], width, ff)
    return w + 4 * width + 8 * n * width, 6 * n * ff * width


def work(case):
    c, k = case, case["kind"]
    if k == "attn":
        return _add(_attn_work(c["heads"], c["kv_heads"], c["head_dim"], c["n"], c["pos0"],
                               4 if c["cache"] == "f32" else 2))
    if k == "batch":
        return _add(*[_attn_work(c["heads"], c["kv_heads"], c["head_dim"], 1, p, 4) for p in _lengths(c)])
    if k == "proj":
        return _add(_matmul_work(c["wtype"], c["q_rows"] + 2 * c["kv_rows"], c["width"], c["n"]))
    if k == "mlp":
        return _add(_mlp_work(c, c["width"]))
    if k == "head":
        return _add(_matmul_work(c["wtype"], c["vocab"], c["width"], c["n"]))
    q, kv, n = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["n"]
    cache = 8 * kv * (c["pos0"] + n)
    attn = (cache, _attn_work(c["heads"], c["kv_heads"], c["head_dim"], n, c["pos0"], 4)[1])
    proj = (_wbytes(c["wtype"], 2 * q + 2 * kv, q), 2 * n * (2 * q + 2 * kv) * q)
    mlp = _mlp_work(c, q)
    layer = (attn[0] + proj[0] + mlp[0] - 8 * n * q, attn[1] + proj[1] + mlp[1])
    return _add(*[layer] * c["layers"], _matmul_work(c["down_type"], c["vocab"], q, 1))


# ---- inputs ----

_be = None


def _backend():
    """The program's backend: one, with its scratch reserved for the largest of these calls."""
    global _be
    if _be is None:
        _be = nibble_amd.HipBackend(0)
        _be.reserve(131072 + 1024, 32, 8192, 8192)
    return _be


class Buffer:
    """A device buffer of the backend, given back with the last of its users: torch keeps this object alive for as
    long as a view of it is."""

    def __init__(self, be, shape, dtype):
        count = math.prod(shape)
        self.be, self.ptr = be, be.alloc(count if dtype == torch.float32 else (count + 1) // 2)
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4" if dtype == torch.float32 else "<f2",
                                         "data": (int(self.ptr), False), "version": 2}

    def __del__(self):
        if self.be is not None:
            self.be.free(self.ptr)


class State:
    """Buffers and weights of one prepared case."""

    def __init__(self, case):
        self.be, self.case, self.held = _backend(), case, []

    def buf(self, *shape, dtype=torch.float32):
        """A device buffer and torch's view of it."""
        b = Buffer(self.be, shape, dtype)
        self.held.append(b)
        return b.ptr, torch.as_tensor(b, device=DEV)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _acts(g, n, width):
    """A residual stream: normal values, one channel in 64 eight times as large."""
    x = _normal(g, n, width)
    x[:, ::64] *= 8
    return x


def _blocks(g, wtype, rows, width):
    """Raw blocks [count, bytes] of a quantized weight: quants of every value, the scales those of a trained weight's
    (elements of about 1 / sqrt(width)), sub-block minimums at the middle of the quants' range."""
    _, be, bb = TYPES[wtype]
    count = rows * width // be
    raw = torch.randint(0, 256, (count, bb), generator=g, device=DEV, dtype=torch.uint8)
    std = width ** -0.5
    rms = {"q4_0": 4.6, "q5_0": 9.2, "q8_0": 74.0, "q4_k": 4.6 * 41, "q5_k": 9.2 * 41, "q6_k": 18.5 * 60}[wtype]
    d = std / rms * (0.5 + torch.rand(count, generator=g, device=DEV))

    def put(at, v):
        raw[:, at:at + 2] = v.to(torch.float16).view(torch.uint8).reshape(count, 2)

    if wtype in ("q4_k", "q5_k"):
        s = torch.randint(16, 64, (count, 8), generator=g, device=DEV, dtype=torch.int32)  # scale = minimum
        put(0, d)
        put(2, d * (7.5 if wtype == "q4_k" else 15.5))
        b = torch.empty(count, 12, device=DEV, dtype=torch.int32)
        b[:, 0:4] = s[:, :4] | ((s[:, 4:] >> 4) << 6)
        b[:, 4:8] = b[:, 0:4]
        b[:, 8:12] = (s[:, 4:] & 15) | ((s[:, 4:] & 15) << 4)
        raw[:, 4:16] = b.to(torch.uint8)
    elif wtype == "q6_k":
        s = torch.randint(24, 97, (count, 16), generator=g, device=DEV, dtype=torch.int32)
        s = torch.where(torch.rand(count, 16, generator=g, device=DEV) < 0.5, -s, s)
        raw[:, 192:208] = s.to(torch.int8).view(torch.uint8)
        put(208, d)
    else:
        put(0, d)
    return raw


def _raw_weight(g, wtype, rows, width):
    if wtype in ("f32", "f16"):
        return (_normal(g, rows, width) * width ** -0.5).to(torch.float32 if wtype == "f32" else torch.float16)
    return _blocks(g, wtype, rows, width)


def _tensor(raw, wtype, rows, width):
    """The weight as a program holds it: a view of host memory, of which the backend keeps a copy on the device."""
    host = np.ascontiguousarray(raw.cpu().numpy())
    if wtype in ("f32", "f16"):
        return nibble_amd.weight(host)
    return nibble_amd.weight(host.reshape(-1), shape=(rows, width), dtype=TYPES[wtype][0])


_held = []  # host arrays whose device copies the backend keeps by their address


def _weight(g, wtype, rows, width):
    t = _tensor(_raw_weight(g, wtype, rows, width), wtype, rows, width)
    _held.append(t)
    return t


def _norm_weight(g, width):
    return 0.8 + 0.4 * torch.rand(width, generator=g, device=DEV)


def _vector(v):
    t = nibble_amd.weight(np.ascontiguousarray(v.cpu().numpy()))
    _held.append(t)
    return t


def _factors(c):
    return synth.llama3_freq_factors(c["head_dim"], c["base"]) if c["llama3"] else None


# The inputs of each kind, in the order that both prepare() and exact() draw them.

def _attn_inputs(c, g, n, pos0):
    h, kv, hd = c["heads"], c["kv_heads"], c["head_dim"]
    return (_normal(g, n, h, hd), _normal(g, n, kv, hd), _normal(g, n, kv, hd), _normal(g, pos0, kv, hd),
            _normal(g, pos0, kv, hd))


def _batch_inputs(c, g):
    """Per sequence as _attn_inputs, with 1 % of the cached K rows eight times as large."""
    for length in _lengths(c):
        q, k, v, ck, cv = _attn_inputs(c, g, 1, length)
        ck[37::100] *= 8
        yield q, k, v, ck, cv


def _proj_shapes(c):
    return [c["q_rows"], c["kv_rows"], c["kv_rows"]]


def _layer_shapes(c):
    q, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    w, d = c["wtype"], c["down_type"]
    return {"wq": (w, q, q), "wk": (w, kv, q), "wv": (w, kv, q), "wo": (w, q, q), "gate": (w, c["ff"], q),
            "up": (w, c["ff"], q), "down": (d, q, c["ff"])}


def _model_inputs(c, g):
    """Embedding table (also the head), per layer (norms, weights, cached K and V rows), last norm, token ids."""
    q = c["heads"] * c["head_dim"]
    table = _raw_weight(g, c["down_type"], c["vocab"], q)
    layers = []
    for _ in range(c["layers"]):
        layer = {k: _raw_weight(g, *s) for k, s in _layer_shapes(c).items()}
        layer.update(norm1=_norm_weight(g, q), norm2=_norm_weight(g, q),
                     k=_normal(g, c["pos0"], c["kv_heads"], c["head_dim"]),
                     v=_normal(g, c["pos0"], c["kv_heads"], c["head_dim"]))
        layers.append(layer)
    ids = torch.randint(0, c["vocab"], (c["n"],), generator=g, device=DEV)
    return table, layers, _norm_weight(g, q), ids


def prepare(case, seed):
    c, s, g = case, State(case), _gen(seed)
    be, k = s.be, case["kind"]
    be.sync()
    fill = []  # (view, values)
    if k == "attn":
        h, kv, hd, n, pos0 = c["heads"], c["kv_heads"], c["head_dim"], c["n"], c["pos0"]
        q, kn, vn, ck, cv = _attn_inputs(c, g, n, pos0)
        dt = torch.float32 if c["cache"] == "f32" else torch.float16
        s.q, a = s.buf(n, h, hd)
        s.k_new, b = s.buf(n, kv, hd)
        s.v_new, d = s.buf(n, kv, hd)
        s.k, s.k_view = s.buf(pos0 + n, kv, hd, dtype=dt)
        s.v, s.v_view = s.buf(pos0 + n, kv, hd, dtype=dt)
        s.out, s.out_view = s.buf(n, h, hd)
        s.factors = _factors(c)
        fill += [(a, q), (b, kn), (d, vn), (s.k_view[:pos0], ck), (s.v_view[:pos0], cv)]
        be.reserve_rope(hd, c["base"], c["neox"], s.factors)
    elif k == "batch":
        h, kv, hd = c["heads"], c["kv_heads"], c["head_dim"]
        s.pos = _lengths(c)
        s.q, s.k, s.v, s.k_new, s.v_new, s.out = [], [], [], [], [], []
        s.rows = []
        ob, s.out_view = s.buf(c["n_seq"], h, hd)
        be.sync()
        for i, (q, kn, vn, ck, cv) in enumerate(_batch_inputs(c, g)):
            p = s.pos[i]
            views = []
            for lst, shape in ((s.q, (1, h, hd)), (s.k_new, (1, kv, hd)), (s.v_new, (1, kv, hd)),
                               (s.k, (p + 1, kv, hd)), (s.v, (p + 1, kv, hd))):
                ptr, view = s.buf(*shape)
                lst.append(ptr)
                views.append(view)
            s.out.append(ob.at(i * h * hd))
            be.sync()
            for view, val in zip(views, (q, kn, vn)):
                view.copy_(val)
            views[3][:p].copy_(ck)
            views[4][:p].copy_(cv)
            s.rows.append((views[3][p], views[4][p]))
        s.factors = _factors(c)
        be.reserve_rope(hd, c["base"], c["neox"], s.factors)
    elif k == "proj":
        n, width = c["n"], c["width"]
        s.x, a = s.buf(n, width)
        fill.append((a, _acts(g, n, width)))
        s.w = [_weight(g, c["wtype"], r, width) for r in _proj_shapes(c)]
        s.b = [_vector(_normal(g, r)) for r in _proj_shapes(c)] if c["bias"] else None
        outs = [s.buf(n, r) for r in _proj_shapes(c)]
        s.y, s.views = [o[0] for o in outs], [o[1] for o in outs]
    elif k == "mlp":
        n, width, ff = c["n"], c["width"], c["ff"]
        s.x, a = s.buf(n, width)
        fill.append((a, _acts(g, n, width)))
        s.norm = _vector(_norm_weight(g, width))
        s.gate_w, s.up_w = _weight(g, c["wtype"], ff, width), _weight(g, c["wtype"], ff, width)
        s.down_w = _weight(g, c["down_type"], width, ff)
        s.h, _ = s.buf(n, width)
        (s.gate, _), (s.up, _) = s.buf(n, ff), s.buf(n, ff)
        s.out, s.out_view = s.buf(n, width)
    elif k == "head":
        n, width = c["n"], c["width"]
        s.x, a = s.buf(n, width)
        fill.append((a, _acts(g, n, width)))
        s.norm = _vector(_norm_weight(g, width))
        s.w = _weight(g, c["wtype"], c["vocab"], width)
        s.h, _ = s.buf(n, width)
        s.out, s.out_view = s.buf(n, c["vocab"])
    else:
        n, pos0, kv, hd = c["n"], c["pos0"], c["kv_heads"], c["head_dim"]
        width = c["heads"] * hd
        table, layers, last, ids = _model_inputs(c, g)
        s.table = _tensor(table, c["down_type"], c["vocab"], width)
        _held.append(s.table)
        s.last_norm, s.ids = _vector(last), ids.cpu().numpy().astype(np.int32)
        s.layers = []
        for layer in layers:
            out = {}
            for name, (t, rows, w) in _layer_shapes(c).items():
                out[name] = _tensor(layer[name], t, rows, w)
                _held.append(out[name])
            out["norm1"], out["norm2"] = _vector(layer["norm1"]), _vector(layer["norm2"])
            out["k"], kview = s.buf(pos0 + n, kv, hd)
            out["v"], vview = s.buf(pos0 + n, kv, hd)
            fill += [(kview[:pos0], layer["k"]), (vview[:pos0], layer["v"])]
            s.layers.append((out, kview[pos0:], vview[pos0:]))
        for name, w in (("x", width), ("h", width), ("q", width), ("attn", width), ("gate", c["ff"]), ("up", c["ff"])):
            setattr(s, name, s.buf(n, w)[0])
        s.k_new, s.v_new = s.buf(n, kv * hd)[0], s.buf(n, kv * hd)[0]
        s.last = s.buf(width)[0]
        s.logits, s.logits_view = s.buf(c["vocab"])
        s.factors = _factors(c)
        be.reserve_rope(hd, c["base"], c["neox"], s.factors)
    be.sync()
    for view, val in fill:
        view.copy_(val)
    torch.cuda.synchronize()
    if k in ("proj", "mlp", "head", "model"):
        run(s)  # the program's model is loaded: the weights are on the device
        be.sync()
    return s


# ---- the passes ----

def _mlp(be, s, x, norm, gate_w, up_w, down_w, h, out, n, width, ff):
    """out = x + down(silu(gate(norm(x))) * up(norm(x)))."""
    be.rmsnorm(x, norm, h, n, EPS)
    be.matmul_multi([gate_w, up_w], h, [s.gate, s.up], n)
    be.silu_mul(s.gate, s.up, n * ff)
    be.matmul(down_w, s.gate, out, n)
    be.add(out, x, n * width)


def run(state):
    s, c, be = state, state.case, state.be
    k = c["kind"]
    if k == "attn":
        f = be.append_rope_attention if c["cache"] == "f32" else be.append_rope_attention_f16kv
        f(s.q, s.k, s.v, s.k_new, s.v_new, s.out, c["n"], c["pos0"], c["heads"], c["kv_heads"], c["head_dim"],
          c["base"], c["neox"], s.factors)
        return {"out": s.out_view, "k": s.k_view[c["pos0"]:], "v": s.v_view[c["pos0"]:]}
    if k == "batch":
        be.append_rope_attention_batch(s.q, s.k, s.v, s.k_new, s.v_new, s.out, s.pos, c["heads"], c["kv_heads"],
                                       c["head_dim"], c["base"], c["neox"], s.factors)
        return {"out": s.out_view, "k": [r[0] for r in s.rows], "v": [r[1] for r in s.rows]}
    if k == "proj":
        be.matmul_multi(s.w, s.x, s.y, c["n"])
        if s.b is not None:
            for y, b in zip(s.y, s.b):
                be.add_bias(y, b, c["n"])
        return s.views
    if k == "mlp":
        _mlp(be, s, s.x, s.norm, s.gate_w, s.up_w, s.down_w, s.h, s.out, c["n"], c["width"], c["ff"])
        return s.out_view
    if k == "head":
        be.rmsnorm(s.x, s.norm, s.h, c["n"], EPS)
        be.matmul(s.w, s.h, s.out, c["n"])
        return s.out_view
    n, pos0, hd, width = c["n"], c["pos0"], c["head_dim"], c["heads"] * c["head_dim"]
    be.embed(s.table, s.ids, s.x)
    for w, _, _ in s.layers:
        be.rmsnorm(s.x, w["norm1"], s.h, n, EPS)
        be.matmul_multi([w["wq"], w["wk"], w["wv"]], s.h, [s.q, s.k_new, s.v_new], n)
        be.append_rope_attention(s.q, w["k"], w["v"], s.k_new, s.v_new, s.attn, n, pos0, c["heads"], c["kv_heads"],
                                 hd, c["base"], c["neox"], s.factors)
        be.matmul(w["wo"], s.attn, s.h, n)
        be.add(s.x, s.h, n * width)
        _mlp(be, s, s.x, w["norm2"], w["gate"], w["up"], w["down"], s.h, s.q, n, width, c["ff"])
        s.x, s.q = s.q, s.x
    be.rmsnorm(s.x.at((n - 1) * width), s.last_norm, s.last, 1, EPS)
    be.matmul(s.table, s.last, s.logits, 1)
    return {"logits": s.logits_view, "k": [r[1] for r in s.layers], "v": [r[2] for r in s.layers]}


# ---- tolerance ----

def tolerance(case):
    """About four times what two correct implementations differ by, as measured: fp32 attention (n <= 16) and F16
    projections are 1e-7..5e-7 from exact() (max 4e-6); on fp16 operands a prompt's attention is 5e-4 from it (max
    5e-3); an appended fp16 row differs by a unit in the last place where its fp32 value sits at a tie. A quantized
    matmul has one right answer (integer dots, the format's float sums in block order), so projections are exact. In a
    block or a model a last-bit difference of a norm, an exponential or an attention sum can move an activation over a
    rounding boundary of the 8-bit activation formats: a block whose input moves by units in the last place differs
    by 3.3e-4 (max 0.014), a model whose attention runs in fp32 by 0.022 (max 0.09)."""
    k = case["kind"]
    if k in ("attn", "batch"):
        if k == "attn" and case["n"] > 16:
            return {"rel": 2e-3, "max": 0.02}
        return {"rel": 2e-4, "max": 2e-3} if case.get("cache") == "f16" else {"rel": 2e-6, "max": 2e-5}
    wtypes = {case["wtype"], case.get("down_type", case["wtype"])}
    if k == "model":
        return {"rel": 5e-3, "max": 0.1} if case["n"] <= 16 else {"rel": 0.03, "max": 0.4}
    if wtypes == {"f16"}:
        return {"rel": 2e-6, "max": 1.5e-5}
    return "exact" if k == "proj" else {"rel": 1.5e-3, "max": 0.06}


# ---- the same in 64 bits ----

def _dequant(raw, wtype, rows, width):
    """The weight [rows, width] that a raw weight stands for (the block formats of ggml)."""
    if wtype in ("f32", "f16"):
        return raw.double()
    b = raw.to(torch.int32)
    count = b.shape[0]

    def half(at):
        return raw[:, at:at + 2].contiguous().view(torch.float16).double()

    if wtype == "q8_0":
        w = half(0) * raw[:, 2:].contiguous().view(torch.int8).double()
    elif wtype in ("q4_0", "q5_0"):
        qs = b[:, -16:]
        q = torch.cat([qs & 15, qs >> 4], 1)
        if wtype == "q5_0":
            bit = torch.arange(32, device=b.device)
            q = q + (((b[:, 2:6].gather(1, (bit // 8).expand(count, 32))) >> (bit % 8)) & 1) * 16
        w = half(0) * (q - (8 if wtype == "q4_0" else 16)).double()
    elif wtype in ("q4_k", "q5_k"):
        p = b[:, 4:16]
        sc = torch.cat([p[:, :4] & 63, (p[:, 8:] & 15) | ((p[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, -128:].reshape(count, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(count, 8, 32)
        if wtype == "q5_k":
            q = q + ((b[:, 16:48].reshape(count, 1, 32) >> torch.arange(8, device=b.device).reshape(1, 8, 1)) & 1) * 16
        w = (half(0) * sc).unsqueeze(2) * q - (half(2) * mn).unsqueeze(2)
    else:
        ql, qh = b[:, :128].reshape(count, 2, 2, 32), b[:, 128:192].reshape(count, 2, 1, 32)
        lo = torch.stack([ql & 15, ql >> 4], 2).reshape(count, 2, 4, 32)
        q = (lo | (((qh >> (2 * torch.arange(4, device=b.device)).reshape(1, 1, 4, 1)) & 3) << 4)) - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double()
        w = half(208).unsqueeze(2) * sc.unsqueeze(2) * q.reshape(count, 16, 16)
    return w.reshape(rows, width)


def _matmul64(raw, wtype, rows, x):
    """x [n, width] times the weight's transpose, in slices of rows."""
    _, be, _ = TYPES[wtype]
    width, per = x.shape[1], 1 if TYPES[wtype][1] == 1 else x.shape[1] // be
    out = []
    for r0 in range(0, rows, 16384):
        r1 = min(rows, r0 + 16384)
        out.append(x @ _dequant(raw[r0 * per:r1 * per], wtype, r1 - r0, width).T.contiguous())
    return torch.cat(out, 1)


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos0, c):
    n, _, hd = x.shape
    x = x.double()
    inv = float(np.float32(c["base"])) ** (-2.0 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)
    th = (pos0 + torch.arange(n, device=x.device, dtype=torch.float64)).reshape(n, 1) * inv
    if c["llama3"]:
        th = th / torch.from_numpy(_factors(c)).to(x.device).double()
    cos, sin = torch.cos(th).unsqueeze(1), torch.sin(th).unsqueeze(1)
    a, b = (x[..., :hd // 2], x[..., hd // 2:]) if c["neox"] else (x[..., 0::2], x[..., 1::2])
    ra, rb = a * cos - b * sin, a * sin + b * cos
    return torch.cat([ra, rb], -1) if c["neox"] else torch.stack([ra, rb], -1).reshape(x.shape)


def _attn64(q, k, v, pos0):
    """q [n, H, D] (rotated) over k, v [pos0 + n, KV, D]: causal softmax attention, a head and 1024 rows at a time."""
    n, h, hd = q.shape
    group = h // k.shape[1]
    out = torch.empty(n, h, hd, device=q.device, dtype=torch.float64)
    for i in range(h):
        kt, vi = k[:, i // group].double().T.contiguous(), v[:, i // group].double().contiguous()
        for t0 in range(0, n, 1024):
            t1 = min(n, t0 + 1024)
            keys = pos0 + t1
            sc = (q[t0:t1, i].contiguous() @ kt[:, :keys].contiguous()) * hd ** -0.5
            at = torch.arange(keys, device=q.device)
            sc.masked_fill_(at > pos0 + torch.arange(t0, t1, device=q.device).unsqueeze(1), -math.inf)
            out[t0:t1, i] = torch.softmax(sc, 1) @ vi[:keys]
    return out


def _layer_attn64(c, q, kn, vn, ck, cv, pos0, f16):
    """Attention of the new rows over the cache with them appended (as it holds them), and the appended rows."""
    kr = _rope64(kn, pos0, c)
    kc, vc = (torch.cat([ck.half(), kr.half()]), torch.cat([cv.half(), vn.half()])) if f16 else \
        (torch.cat([ck.double(), kr]), torch.cat([cv.double(), vn.double()]))
    return _attn64(_rope64(q, pos0, c), kc, vc, pos0), kr, vn


def _mlp64(x, norm, gate, up, down, wtype, down_type, ff):
    h = _norm64(x, norm)
    a, b = _matmul64(gate, wtype, ff, h), _matmul64(up, wtype, ff, h)
    return x + _matmul64(down, down_type, x.shape[1], a * torch.sigmoid(a) * b)


def exact(case, seed):
    c, g, k = case, _gen(seed), case["kind"]
    if k == "attn":
        q, kn, vn, ck, cv = _attn_inputs(c, g, c["n"], c["pos0"])
        f16 = c["cache"] == "f16"
        out, kr, vr = _layer_attn64(c, q, kn, vn, ck, cv, c["pos0"], f16)
        return {"out": out, "k": kr, "v": vr.double()}
    if k == "batch":
        outs, ks, vs = [], [], []
        for p, (q, kn, vn, ck, cv) in zip(_lengths(c), _batch_inputs(c, g)):
            o, kr, vr = _layer_attn64(c, q, kn, vn, ck, cv, p, False)
            outs.append(o)
            ks.append(kr[0])
            vs.append(vr[0].double())
        return {"out": torch.cat(outs), "k": ks, "v": vs}
    if k == "proj":
        x = _acts(g, c["n"], c["width"]).double()
        ws = [_raw_weight(g, c["wtype"], r, c["width"]) for r in _proj_shapes(c)]
        bs = [_normal(g, r).double() for r in _proj_shapes(c)] if c["bias"] else [0.0] * 3
        return [_matmul64(w, c["wtype"], r, x) + b for w, r, b in zip(ws, _proj_shapes(c), bs)]
    if k in ("mlp", "head"):
        x = _acts(g, c["n"], c["width"]).double()
        norm = _norm_weight(g, c["width"])
        if k == "head":
            table = _raw_weight(g, c["wtype"], c["vocab"], c["width"])
            return _matmul64(table, c["wtype"], c["vocab"], _norm64(x, norm))
        ws = [_raw_weight(g, c["wtype"], c["ff"], c["width"]) for _ in range(2)]
        ws.append(_raw_weight(g, c["down_type"], c["width"], c["ff"]))
        return _mlp64(x, norm, *ws, c["wtype"], c["down_type"], c["ff"])
    n, pos0, hd = c["n"], c["pos0"], c["head_dim"]
    width, kv = c["heads"] * hd, c["kv_heads"]
    table, layers, last, ids = _model_inputs(c, g)
    rows = table[ids] if TYPES[c["down_type"]][1] == 1 else \
        table.reshape(c["vocab"], -1, table.shape[1])[ids].reshape(-1, table.shape[1])
    x, ks, vs = _dequant(rows, c["down_type"], n, width), [], []
    shapes = _layer_shapes(c)
    for w in layers:
        def mm(name, v):
            return _matmul64(w[name], shapes[name][0], shapes[name][1], v)
        h = _norm64(x, w["norm1"])
        kn, vn = mm("wk", h).reshape(n, kv, hd), mm("wv", h).reshape(n, kv, hd)
        o, kr, vr = _layer_attn64(c, mm("wq", h).reshape(n, c["heads"], hd), kn, vn, w["k"], w["v"], pos0, False)
        ks.append(kr)
        vs.append(vr)
        x = x + mm("wo", o.reshape(n, width))
        x = _mlp64(x, w["norm2"], w["gate"], w["up"], w["down"], c["wtype"], c["down_type"], c["ff"])
    return {"logits": _matmul64(table, c["down_type"], c["vocab"], _norm64(x[-1:], last))[0], "k": ks, "v": vs}

"""The measured work of this framework: what a program that runs a static-lm
model on one GPU has it do, through the public binding.

Kinds of case
  decode    one token of attention through `layers` KV caches at position `pos`
            (AttentionContext.decode_dev)
  prefill   `n` rows of causal attention from row `start` through `layers`
            caches (AttentionContext.prefill_dev)
  project   a Q4_0 projection of `batch` rows, with the residual add where
            `residual` is set (gemm_q4_0_dev, gemm_q4_0_residual_dev)
  layer     `n` rows through `layers` whole transformer blocks from row
            `start` (layer_forward_dev); n = 1 is a decode step
  model     a prompt of `n` tokens, then `steps` single tokens, with every
            call's logits (model_prefill_dev, model_forward_token_dev)

Attention inputs: v is N(0, 0.5), q and k give scores a few nats apart, as
trained heads do.  Weights are N(0, 1/cols) rounded to Q4_0 by its own rule.
"""
import ctypes
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

EPS = 1e-5


def _product():
    name = "static_lm_amd"
    if name not in sys.modules:
        root = Path.cwd() / "static-lm_amd"
        spec = importlib.util.spec_from_file_location(name, root / "__init__.py",
                                                      submodule_search_locations=[str(root)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# (dim, heads, kv_heads, rope theta, hidden): the attention shapes of the
# repository's configurations and parity tests, one or more of every head_dim
SHAPES = {
    "hd16": (64, 4, 4, 1e4, 192),
    "hd32": (256, 8, 2, 1e4, 704),
    "hd48": (288, 6, 6, 1e4, 768),        # Stories-15M shape
    "hd64": (576, 9, 3, 1e5, 1536),       # SmolLM2-135M shape
    "hd64_mha": (256, 4, 4, 1e4, 704),
    "hd96": (768, 8, 8, 1e4, 2048),
    "hd128": (4096, 32, 8, 5e5, 14336),   # Llama-3-8B shape
    "hd128_gqa8": (2048, 16, 2, 1e5, 5632),
    "hd256": (1024, 4, 4, 1e4, 2816),
}


def listed():
    return [
        # the smallest call a chat with a tiny model makes, over and over:
        # one token, six layers, a short history (launches and latency)
        {"name": "decode_hd48_pos79", "kind": "decode", "shape": "hd48", "layers": 6, "pos": 79},
        # a small model answering: one token through its thirty caches
        {"name": "decode_hd64_pos700", "kind": "decode", "shape": "hd64", "layers": 30,
         "pos": 700},
        # a large model with a few thousand tokens of history
        {"name": "decode_hd128_pos4222", "kind": "decode", "shape": "hd128", "layers": 8,
         "pos": 4222},
        # long documents: the caches stream from HBM
        {"name": "decode_hd128_pos32767", "kind": "decode", "shape": "hd128", "layers": 8,
         "pos": 32767},
        # a one-line prompt of a tiny model
        {"name": "prefill_hd48_n16", "kind": "prefill", "shape": "hd48", "layers": 6,
         "start": 0, "n": 16},
        # an ordinary prompt of a small model
        {"name": "prefill_hd64_n512", "kind": "prefill", "shape": "hd64", "layers": 30,
         "start": 0, "n": 512},
        # a long prompt of a large model
        {"name": "prefill_hd128_n4096", "kind": "prefill", "shape": "hd128", "layers": 1,
         "start": 0, "n": 4096},
        # the next turn of a conversation: an odd number of rows behind a history
        {"name": "prefill_hd128_s1000_n777", "kind": "prefill", "shape": "hd128", "layers": 1,
         "start": 1000, "n": 777},
        # the output projection of a short prompt (few rows, every weight read)
        {"name": "project_4096x4096_b12", "kind": "project", "rows": 4096, "cols": 4096,
         "batch": 12, "residual": True},
        # a large model's decode step, weights and caches together
        {"name": "layer_hd128_pos599", "kind": "layer", "shape": "hd128", "layers": 4,
         "start": 599, "n": 1},
        # a large model's prompt: projections, attention, FFN
        {"name": "layer_hd128_n2048", "kind": "layer", "shape": "hd128", "layers": 1,
         "start": 0, "n": 2048},
        # a whole small model: a prompt, then its first tokens
        {"name": "model_hd64_n130", "kind": "model", "shape": "hd64", "layers": 30,
         "vocab": 49152, "n": 130, "steps": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "project", "layer", "model"])
    if kind == "project":
        rows, cols = rng.choice([(4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336),
                                 (576, 576), (1536, 576), (576, 1536), (288, 768)])
        return {"kind": kind, "rows": rows, "cols": cols, "batch": _log(rng, 1, 2048),
                "residual": rng.random() < 0.5}
    shape = rng.choice(sorted(SHAPES))
    dim, heads, kvh = SHAPES[shape][:3]
    kvd = dim // heads * kvh
    if kind == "decode":
        layers = rng.choice([2, 6, 8])
        # at most the 32k-row case's cache bytes
        top = min(32768, 8 * 32768 * 1024 // (layers * kvd))
        return {"kind": kind, "shape": shape, "layers": layers, "pos": _log(rng, 2, top) - 1}
    if kind == "prefill":
        layers = rng.choice([1, 2])
        n = _log(rng, 2, 2900 if layers == 2 else 4096)
        start = 0 if rng.random() < 0.6 else _log(rng, 1, max(2, (4096 - n) // 2 + 1))
        return {"kind": kind, "shape": shape, "layers": layers, "start": start, "n": n}
    if kind == "layer":
        one = rng.random() < 0.4
        return {"kind": kind, "shape": shape, "layers": 2 if one else 1,
                "start": _log(rng, 1, 4000) if one or rng.random() < 0.3 else 0,
                "n": 1 if one else _log(rng, 2, 1500)}
    shape = rng.choice([s for s in sorted(SHAPES) if s != "hd128"])
    return {"kind": kind, "shape": shape, "layers": rng.choice([2, 6, 12]),
            "vocab": rng.choice([512, 8191, 32000]), "n": _log(rng, 2, 400),
            "steps": rng.choice([1, 2, 4])}


# ---- inputs ----

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(g, shape, scale):
    return torch.randn(shape, generator=g, device="cuda") * scale


def _q4_blocks(g, rows, cols):
    """A row-major N(0, 1/cols) matrix as Q4_0 blocks [rows * cols / 32, 18]."""
    x = _normal(g, (rows * cols // 32, 32), 1.0 / math.sqrt(cols))
    big = x.gather(1, x.abs().argmax(1, keepdim=True))
    d = big / -8.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = torch.clamp((x * inv + 8.5).to(torch.int32), 0, 15).to(torch.uint8)
    blk = torch.empty((x.shape[0], 18), dtype=torch.uint8, device="cuda")
    blk[:, :2] = d.half().view(torch.uint8).reshape(-1, 2)
    blk[:, 2:] = q[:, :16] | (q[:, 16:] << 4)
    return blk


def _dequant64(blk, rows, cols):
    d = blk[:, :2].contiguous().view(torch.float16).double()
    lo = (blk[:, 2:] & 15).double() - 8
    hi = (blk[:, 2:] >> 4).double() - 8
    return (torch.cat([lo, hi], 1) * d).reshape(rows, cols)


class _KvRegion:
    """The context's KV region [layers][K|V][max_seq_len][kv_dim] for torch;
    keeps the context alive as long as a tensor looks at it."""

    def __init__(self, ctx, layers, msl, kvd):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"shape": (layers, 2, msl, kvd), "typestr": "<f4",
                                         "data": (ctx.kv_device_ptr(), False), "version": 3}


def _max_rows(case):
    if case["kind"] == "decode":
        rows = case["pos"] + 1
    elif case["kind"] == "model":
        rows = case["n"] + case["steps"]
    else:
        rows = case["start"] + case["n"]
    return max(256, (rows + 255) // 256 * 256)


def _context(case):
    P = _product()
    dim, heads, kvh, theta, _ = SHAPES[case["shape"]]
    msl = _max_rows(case)
    ctx = P.AttentionContext(dim, heads, kvh, msl, case["layers"], theta)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    kvd = dim // heads * kvh
    kv = torch.as_tensor(_KvRegion(ctx, case["layers"], msl, kvd), device="cuda")
    return ctx, stream, kv


def _history(case, seed, kv):
    """Cache rows of the earlier turns, as their prefill left them."""
    rows = case["pos"] if case["kind"] == "decode" else case.get("start", 0)
    if rows:
        g = _gen(seed, 1)
        for layer in range(case["layers"]):
            kv[layer, 0, :rows] = _normal(g, (rows, kv.shape[3]), 1.0)
            kv[layer, 1, :rows] = _normal(g, (rows, kv.shape[3]), 0.5)


def _qkv(case, seed):
    dim, heads, kvh = SHAPES[case["shape"]][:3]
    kvd = dim // heads * kvh
    n = case.get("n", 1)
    g = _gen(seed, 2)
    return (_normal(g, (case["layers"], n, dim), 2.0), _normal(g, (case["layers"], n, kvd), 1.0),
            _normal(g, (case["layers"], n, kvd), 0.5))


_MATRICES = ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")


def _matrix_shapes(case):
    dim, heads, kvh, _, hidden = SHAPES[case["shape"]]
    kvd = dim // heads * kvh
    return {"wq": (dim, dim), "wk": (kvd, dim), "wv": (kvd, dim), "wo": (dim, dim),
            "w_gate": (hidden, dim), "w_up": (hidden, dim), "w_down": (dim, hidden)}


def _layer_blocks(case, seed, layer):
    """One layer's Q4_0 blocks and RMSNorm scales, on the GPU."""
    g = _gen(seed, 100 + layer)
    shapes = _matrix_shapes(case)
    dim = SHAPES[case["shape"]][0]
    blocks = {m: _q4_blocks(g, *shapes[m]) for m in _MATRICES}
    norms = [1.0 + _normal(g, (dim,), 0.1) for _ in range(2)]
    return blocks, norms


def _layer_weights(case, seed):
    P = _product()
    shapes = _matrix_shapes(case)
    out, keep = [], []
    for layer in range(case["layers"]):
        blocks, norms = _layer_blocks(case, seed, layer)
        mats = [P.Q4Matrix(blocks[m].cpu().numpy(), *shapes[m]) for m in _MATRICES]
        out.append(P.LayerWeights(norms[0].data_ptr(), *mats[:4], norms[1].data_ptr(), *mats[4:]))
        keep.append(norms)
    return out, keep


def _tokens(case, seed):
    rng = np.random.default_rng([seed, 7])
    return rng.integers(0, case["vocab"], case["n"] + case["steps"]).astype(np.int32)


def _model_blocks(case, seed):
    dim = SHAPES[case["shape"]][0]
    g = _gen(seed, 50)
    emb = _q4_blocks(g, case["vocab"], dim)
    head = _q4_blocks(g, case["vocab"], dim)
    return emb, head, 1.0 + _normal(g, (dim,), 0.1)


def prepare(case, seed):
    P = _product()
    kind = case["kind"]
    s = {"case": case}
    if kind == "project":
        g = _gen(seed, 3)
        rows, cols, batch = case["rows"], case["cols"], case["batch"]
        s["w"] = P.Q4Matrix(_q4_blocks(g, rows, cols).cpu().numpy(), rows, cols)
        s["x"] = _normal(g, (batch, cols), 1.0)
        s["res"] = _normal(g, (batch, rows), 1.0) if case["residual"] else None
        s["out"] = torch.empty((batch, rows), device="cuda")
        # projections take a context for its stream and scratch
        s["ctx"] = P.AttentionContext(64, 2, 2, 256, 1)
        s["stream"] = torch.cuda.Stream()
        s["ctx"].set_stream(s["stream"].cuda_stream)
        torch.cuda.synchronize()
        return s
    s["ctx"], s["stream"], kv = _context(case)
    if kind in ("decode", "prefill"):
        _history(case, seed, kv)
        s["q"], s["k"], s["v"] = _qkv(case, seed)
        s["out"] = torch.empty_like(s["q"])
        a = case["pos"] if kind == "decode" else case["start"]
        s["rows"] = kv[:, :, a:a + s["q"].shape[1]]
    elif kind == "layer":
        _history(case, seed, kv)
        s["weights"], s["keep"] = _layer_weights(case, seed)
        dim = SHAPES[case["shape"]][0]
        s["x0"] = _normal(_gen(seed, 2), (case["n"], dim), 1.0)
        s["x"] = torch.empty_like(s["x0"])
    else:
        layers, s["keep"] = _layer_weights(case, seed)
        emb, head, norm = _model_blocks(case, seed)
        dim = SHAPES[case["shape"]][0]
        s["norm"] = norm
        s["weights"] = P.ModelWeights(P.Q4Matrix(emb.cpu().numpy(), case["vocab"], dim), layers,
                                      norm.data_ptr(),
                                      P.Q4Matrix(head.cpu().numpy(), case["vocab"], dim))
        s["tokens"] = _tokens(case, seed)
        s["logits"] = torch.empty((1 + case["steps"], case["vocab"]), device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "project":
        x, out = s["x"].data_ptr(), s["out"].data_ptr()
        if s["res"] is not None:
            ctx.gemm_q4_0_residual_dev(s["w"], x, case["batch"], s["res"].data_ptr(), out)
        else:
            ctx.gemm_q4_0_dev(s["w"], x, case["batch"], out)
        return s["out"]
    if kind in ("decode", "prefill"):
        q, k, v, out = s["q"], s["k"], s["v"], s["out"]
        n, dim, kvd = q.shape[1], q.shape[2], k.shape[2]
        pq, pk, pv, po = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
        for layer in range(case["layers"]):
            a, b = 4 * layer * n * dim, 4 * layer * n * kvd
            if kind == "decode":
                ctx.decode_dev(layer, case["pos"], pq + a, pk + b, pv + b, po + a)
            else:
                ctx.prefill_dev(layer, case["start"], n, pq + a, pk + b, pv + b, po + a)
        return {"out": out, "kv": s["rows"]}
    if kind == "layer":
        with torch.cuda.stream(s["stream"]):
            s["x"].copy_(s["x0"])  # the block works in place on the residual stream
        for layer in range(case["layers"]):
            ctx.layer_forward_dev(layer, case["start"], case["n"], s["weights"][layer], EPS,
                                  s["x"].data_ptr())
        return s["x"]
    n, toks, logits = case["n"], s["tokens"], s["logits"]
    row = 4 * case["vocab"]
    ctx.model_prefill_dev(s["weights"], EPS, toks[:n], 0, logits.data_ptr())
    for i in range(case["steps"]):
        ctx.model_forward_token_dev(s["weights"], EPS, int(toks[n + i]), n + i,
                                    logits.data_ptr() + (1 + i) * row)
    return logits


# ---- what a pass cannot do without ----

def _attention_work(case, start, n, layers):
    dim, heads, kvh = SHAPES[case["shape"]][:3]
    hd = dim // heads
    kvd = hd * kvh
    pairs = n * start + n * (n + 1) // 2
    return {"bytes": layers * 4 * (2 * (start + n) * kvd + 2 * n * dim + 2 * n * kvd),
            "flops": layers * 4 * hd * heads * pairs}


def work(case):
    kind = case["kind"]
    if kind == "project":
        r, c, b = case["rows"], case["cols"], case["batch"]
        return {"bytes": r * c // 32 * 18 + 4 * b * (c + r * (2 if case["residual"] else 1)),
                "flops": 2 * b * r * c}
    layers = case["layers"]
    if kind == "decode":
        return _attention_work(case, case["pos"], 1, layers)
    if kind == "prefill":
        return _attention_work(case, case["start"], case["n"], layers)
    weights = sum(r * c for r, c in _matrix_shapes(case).values())
    dim = SHAPES[case["shape"]][0]
    if kind == "layer":
        n = case["n"]
        a = _attention_work(case, case["start"], n, layers)
        return {"bytes": layers * weights // 32 * 18 + a["bytes"] + 8 * n * dim,
                "flops": a["flops"] + 2 * n * layers * weights}
    total = {"bytes": 0, "flops": 0}
    calls = [(0, case["n"])] + [(case["n"] + i, 1) for i in range(case["steps"])]
    for start, n in calls:
        a = _attention_work(case, start, n, layers)
        head = case["vocab"] * dim
        total["bytes"] += (layers * weights + head) // 32 * 18 + a["bytes"] + 4 * case["vocab"]
        total["flops"] += a["flops"] + 2 * n * layers * weights + 2 * head
    return total


def tolerance(case):
    kind = case["kind"]
    if kind == "project":
        # f32 sums of cols / 32 block terms
        return {"rel": 2e-6}
    if kind in ("decode", "prefill"):
        # f32 dot products, exponentials and weighted sums
        return {"rel": 4e-6}
    # another order of f32 sums moves an activation across a Q8_0 step now and
    # then, and every later layer carries it on: against the 64-bit evaluation
    # four layers of a large model are 0.7% apart, a whole small model 2.2%
    return {"rel": 3e-2} if kind == "layer" else {"rel": 8e-2}


# ---- the same in 64 bits ----

def _rope64(x, pos0, hd, theta):
    """Interleaved pairs rotated by the tables' f32 angles, in 64 bits."""
    n = x.shape[0]
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    freq = torch.tensor([powf(theta, float(np.float32(j) / np.float32(hd)))
                         for j in range(0, hd, 2)], device="cuda").reciprocal()
    pos = torch.arange(pos0, pos0 + n, device="cuda").float()
    ang = (pos[:, None] * freq[None, :]).double()
    c, sn = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    p = x.reshape(n, -1, hd // 2, 2)
    a, b = p[..., 0], p[..., 1]
    return torch.stack([a * c - b * sn, a * sn + b * c], -1).reshape(n, -1)


def _attend64(q, kc, vc, start, heads, kvh):
    """Causal attention of rotated q [n][dim] at rows start.. over the caches."""
    n, dim = q.shape
    hd = dim // heads
    out = torch.empty_like(q)
    rows = kc.shape[0]
    keys = torch.arange(rows, device="cuda")
    for h in range(heads):
        g = h // (heads // kvh)
        k, v = kc[:, g * hd:(g + 1) * hd], vc[:, g * hd:(g + 1) * hd]
        for b in range(0, n, 1024):
            e = min(n, b + 1024)
            sc = q[b:e, h * hd:(h + 1) * hd] @ k.T / math.sqrt(hd)
            qpos = torch.arange(start + b, start + e, device="cuda")
            sc.masked_fill_(keys[None, :] > qpos[:, None], float("-inf"))
            out[b:e, h * hd:(h + 1) * hd] = torch.softmax(sc, 1) @ v
    return out


def _q8_64(x):
    """Q8_0 of f32-rounded rows, back in 64 bits (the format's own rule)."""
    f = x.float().reshape(-1, 32)
    amax = f.abs().amax(1, keepdim=True)
    d = amax / 127.0
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    y = f * inv
    q = torch.sign(y) * torch.floor(y.abs() + 0.5)
    return (q.double() * d.half().double()).reshape(x.shape)


def _norm64(x, w):
    return x / torch.sqrt(x.square().mean(1, keepdim=True) + EPS) * w.double()


def _block64(case, x, start, blocks, norms, kc, vc):
    """One transformer block of rows start.. over caches kc, vc (written)."""
    dim, heads, kvh, theta, _ = SHAPES[case["shape"]]
    hd = dim // heads
    n = x.shape[0]
    w = {m: _dequant64(blocks[m], *_matrix_shapes(case)[m]) for m in _MATRICES}
    a = _q8_64(_norm64(x, norms[0]))
    kc[start:start + n] = _rope64(a @ w["wk"].T, start, hd, theta)
    vc[start:start + n] = a @ w["wv"].T
    q = _rope64(a @ w["wq"].T, start, hd, theta)
    att = _attend64(q, kc[:start + n], vc[:start + n], start, heads, kvh)
    x = x + _q8_64(att) @ w["wo"].T
    a = _q8_64(_norm64(x, norms[1]))
    gate, up = a @ w["w_gate"].T, a @ w["w_up"].T
    return x + _q8_64(gate * torch.sigmoid(gate) * up) @ w["w_down"].T


def exact(case, seed):
    kind = case["kind"]
    if kind == "project":
        g = _gen(seed, 3)
        rows, cols, batch = case["rows"], case["cols"], case["batch"]
        w = _dequant64(_q4_blocks(g, rows, cols), rows, cols)
        y = _q8_64(_normal(g, (batch, cols), 1.0)) @ w.T
        return y + _normal(g, (batch, rows), 1.0).double() if case["residual"] else y
    dim, heads, kvh, theta, _ = SHAPES[case["shape"]]
    hd, kvd, layers = dim // heads, dim // heads * kvh, case["layers"]
    if kind in ("decode", "prefill"):
        start = case["pos"] if kind == "decode" else case["start"]
        q, k, v = _qkv(case, seed)
        n = q.shape[1]
        hist = torch.empty((layers, 2, start + n, kvd), device="cuda")
        _history(case, seed, hist)
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        rows = torch.empty((layers, 2, n, kvd), dtype=torch.float64, device="cuda")
        for i in range(layers):
            rows[i, 0] = _rope64(k[i].double(), start, hd, theta)
            rows[i, 1] = v[i].double()
            kc = torch.cat([hist[i, 0, :start].double(), rows[i, 0]])
            vc = torch.cat([hist[i, 1, :start].double(), rows[i, 1]])
            out[i] = _attend64(_rope64(q[i].double(), start, hd, theta), kc, vc, start, heads,
                               kvh)
        return {"out": out, "kv": rows}
    rows = _max_rows(case)
    if kind == "layer":
        hist = torch.zeros((layers, 2, rows, kvd), device="cuda")
        _history(case, seed, hist)
        x = _normal(_gen(seed, 2), (case["n"], dim), 1.0).double()
        for i in range(layers):
            blocks, norms = _layer_blocks(case, seed, i)
            x = _block64(case, x, case["start"], blocks, norms, hist[i, 0].double(),
                         hist[i, 1].double())
        return x
    emb, head, norm = _model_blocks(case, seed)
    table, head = _dequant64(emb, case["vocab"], dim), _dequant64(head, case["vocab"], dim)
    toks = torch.from_numpy(_tokens(case, seed)).cuda().long()
    caches = torch.zeros((layers, 2, rows, kvd), dtype=torch.float64, device="cuda")
    out = []
    calls = [(0, case["n"])] + [(case["n"] + i, 1) for i in range(case["steps"])]
    parts = [_layer_blocks(case, seed, i) for i in range(layers)]
    for start, n in calls:
        x = table[toks[start:start + n]]
        for i in range(layers):
            x = _block64(case, x, start, *parts[i], caches[i, 0], caches[i, 1])
        out.append(_q8_64(_norm64(x[-1:], norm)) @ head.T)
    return torch.cat(out)

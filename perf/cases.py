"""The work a program gives this library, as cases to be timed and checked.

Five kinds of call, each through the public entry points of
`qx_amd.runtime`, over as many layers as the program runs back to back:

  step     one Granite token's decode_step in 24 layers (q, k, v in hand)
  block    one token's attention half, norm to residual, in every layer: the
           Granite block with Q4 or fp32 weights, the Qwen block with Q4
  decode   one token of a batch: RoPE + append, then attention, per layer
  prompt   the rows of one prompt (or of a chunk of it, or of a few drafted
           tokens to verify): RoPE + append, then causal attention, per layer
  leaves   commitment hashes of the rows of a batch of caches

A pass is what a program does for one token or one prompt: it opens a graph,
encodes, and finishes it (which waits, as the sampler needs the result);
`replay` cases launch a graph captured once instead, as a launch-bound loop
does.  A pass appends at the same position each time, so it first moves the
cursors back, which is what a rejected draft does and costs no GPU work.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from qx_amd import abi
from qx_amd import runtime as rt

DEV = "cuda:0"
DTYPES = {"f32": (torch.float32, abi.F32), "f16": (torch.float16, abi.F16), "bf16": (torch.bfloat16, abi.BF16),
          "tiered": (torch.float16, abi.I8_TIERED)}
SHAPES = {"granite": (16, 8, 64, abi.SHAPE_GRANITE), "qwen": (32, 4, 128, abi.SHAPE_QWEN3)}
WINDOW = 256  # binary16 rows of a tiered value cache
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "tiered": 1 + 2 / 32}

_CTX = []


def _context():
    if not _CTX:
        _CTX.append(rt.Context(0))
    return _CTX[0]


# ---- the cases ------------------------------------------------------------------

def listed():
    return [
        # A chat's early tokens: short contexts, one small launch per layer.
        {"name": "step-granite-short", "kind": "step", "kd": "f32", "vd": "f16", "position": 100},
        # The shipped model: Q4 projections on the default KV plan (fp32 K, f16 V), far into its context.
        {"name": "block-granite-q4", "kind": "block", "shape": "granite", "weights": "q4", "kd": "f32", "vd": "f16",
         "position": 2900, "replay": True},
        # The same model before quantisation, the 24-layer stack at the end of its context.
        {"name": "block-granite-f32", "kind": "block", "shape": "granite", "weights": "f32", "kd": "f32", "vd": "f32",
         "position": 4095, "replay": False},
        # One user of the larger model over a long document, 48 layers.
        {"name": "block-qwen-q4-long", "kind": "block", "shape": "qwen", "weights": "q4", "kd": "f16", "vd": "f16",
         "position": 32767, "replay": True},
        # Batched serving at its largest: 256 sequences at the end of the context.
        {"name": "decode-granite-256", "kind": "decode", "shape": "granite", "kd": "f16", "vd": "f16",
         "sequences": 256, "position": 4095, "layers": 4},
        # An ordinary serving batch of the larger model, at an odd length.
        {"name": "decode-qwen-16", "kind": "decode", "shape": "qwen", "kd": "bf16", "vd": "bf16", "sequences": 16,
         "position": 2999, "layers": 8},
        # Batched serving with the smaller value format.
        {"name": "decode-granite-tiered", "kind": "decode", "shape": "granite", "kd": "f32", "vd": "tiered",
         "sequences": 64, "position": 3999, "layers": 4},
        # A long prompt of the smaller model on 16-bit caches.
        {"name": "prompt-granite-f16", "kind": "prompt", "shape": "granite", "kd": "f16", "vd": "f16", "start": 0,
         "tokens": 2048, "layers": 8},
        # A prompt of ragged length on the default KV plan, which needs fp32 products.
        {"name": "prompt-granite-f32k", "kind": "prompt", "shape": "granite", "kd": "f32", "vd": "f16", "start": 0,
         "tokens": 1900, "layers": 8},
        # A document given to the larger model.
        {"name": "prompt-qwen-bf16", "kind": "prompt", "shape": "qwen", "kd": "bf16", "vd": "bf16", "start": 0,
         "tokens": 8192, "layers": 2},
        # Five drafted tokens verified over a long context.
        {"name": "verify-qwen", "kind": "prompt", "shape": "qwen", "kd": "bf16", "vd": "bf16", "start": 12000,
         "tokens": 5, "layers": 8},
        # The commitment over every row of a batch of caches.
        {"name": "leaves-granite", "kind": "leaves", "shape": "granite", "kd": "f16", "vd": "f16", "sequences": 16,
         "begin": 0, "count": 4096},
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


GRANITE_PLANS = (("f32", "f16"), ("f32", "f32"), ("f16", "f16"), ("bf16", "bf16"))


def draw(rng):
    kind = rng.choice(("step", "block", "block", "decode", "decode", "prompt", "prompt", "prompt", "leaves"))
    shape = rng.choice(("granite", "qwen"))
    if kind == "step":
        kd, vd = rng.choice(GRANITE_PLANS[:3])
        return {"kind": "step", "kd": kd, "vd": vd, "position": _log_int(rng, 16, 1023)}
    if kind == "block" and shape == "granite":
        kd, vd = rng.choice(GRANITE_PLANS[:3])
        return {"kind": "block", "shape": shape, "weights": rng.choice(("q4", "q4", "f32")), "kd": kd, "vd": vd,
                "position": _log_int(rng, 64, 4095), "replay": rng.random() < 0.5}
    if kind == "block":
        kd = rng.choice(("f16", "bf16"))
        return {"kind": "block", "shape": shape, "weights": "q4", "kd": kd, "vd": kd,
                "position": _log_int(rng, 128, 32000), "replay": rng.random() < 0.5}
    if kind == "decode":
        if shape == "granite":
            kd, vd = rng.choice(GRANITE_PLANS + (("f32", "tiered"),))
        else:
            kd = rng.choice(("f16", "bf16"))
            vd = rng.choice((kd, kd, "tiered"))
        sequences = _log_int(rng, 1, 256 if shape == "granite" else 64)
        layers = 4 if sequences > 32 else 8
        # at most the largest listed batch's cache: 256 x 4096 rows of 2 KiB in 4 layers
        row = (BYTES[kd] + BYTES[vd]) * SHAPES[shape][1] * SHAPES[shape][2]
        most = 4 * 256 * 4096 * 2048 * 0.8 / (row * layers * sequences)
        position = _log_int(rng, 128, int(min(most, 4095 if shape == "granite" else 32000)))
        return {"kind": "decode", "shape": shape, "kd": kd, "vd": vd, "sequences": sequences, "position": position,
                "layers": layers}
    if kind == "prompt":
        few = rng.random() < 0.3  # a few drafted rows; else a prompt or a chunk of one
        if shape == "granite":
            kd, vd = rng.choice(GRANITE_PLANS)
            tokens = rng.randint(2, 8) if few else _log_int(rng, 24, 3000)
            start = _log_int(rng, 64, 4000) if few else rng.choice((0, _log_int(rng, 64, 4000)))
            return {"kind": "prompt", "shape": shape, "kd": kd, "vd": vd, "start": min(start, 4096 - tokens),
                    "tokens": tokens, "layers": 8}
        kd = rng.choice(("f16", "bf16"))
        tokens = rng.randint(2, 8) if few else _log_int(rng, 24, 7000)
        # at most the largest listed prompt's products: 8192 rows over 4096 positions each, in 2 layers
        most = int(2 * 8192 * 4096 * 0.8 / ((2 if tokens > 2000 else 8) * tokens) - tokens / 2)
        start = rng.choice((0, 1)) * _log_int(rng, 64, 24000) if not few else _log_int(rng, 64, 24000)
        return {"kind": "prompt", "shape": shape, "kd": kd, "vd": kd, "start": max(0, min(start, most)),
                "tokens": tokens, "layers": 2 if tokens > 2000 else 8}
    kd = rng.choice(("f16", "bf16", "f32"))
    vd = rng.choice((kd, "f16")) if shape == "granite" and kd == "f32" else "f16" if kd == "f32" else kd
    kd = "f16" if kd == "f32" and shape == "qwen" else kd
    sequences = _log_int(rng, 1, 32)
    begin = rng.randint(0, 200)
    return {"kind": "leaves", "shape": shape, "kd": kd, "vd": vd, "sequences": sequences, "begin": begin,
            "count": _log_int(rng, 64, 4096 - begin)}


# ---- inputs ----------------------------------------------------------------------

class _Draws:
    """Seeded values on the device; the same calls give the same values."""

    def __init__(self, seed, part):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed * 1000003 + part)

    def normal(self, shape, dtype=torch.float32, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=dtype).mul_(std)

    def q4(self, rows, cols, std):
        """Group-32 Q4 weights: codes of a normal's width about 7, one binary16 scale a group."""
        lo, hi = (torch.randn((rows, cols // 2), generator=self.g, device=DEV).mul_(2.5).add_(7).round_()
                  .clamp_(0, 15).to(torch.uint8) for _ in range(2))
        scales = torch.rand((rows, cols // 32), generator=self.g, device=DEV).add_(0.5).mul_(std / 2.5)
        return lo | hi << 4, scales.to(torch.float16)


def _layers(case):
    return {"step": 24, "block": 24 if case.get("shape") == "granite" else 48, "leaves": 1}.get(
        case["kind"]) or case["layers"]


def _dims(case):
    return SHAPES[case.get("shape", "granite")]


def _start(case):
    return case["start"] if case["kind"] == "prompt" else case["position"]


def _past(case, seed, layer):
    """The cached rows of one layer, [sequences][positions][kv heads][d]: values that the cache's types hold."""
    hq, hk, d, _ = _dims(case)
    n = case["begin"] + case["count"] if case["kind"] == "leaves" else _start(case)
    shape = (case.get("sequences", 1), n, hk, d)
    kt, vt = DTYPES[case["kd"]][0], DTYPES[case["vd"]][0]
    r = _Draws(seed, 2 * layer)
    # Granite scales its products by 1/64 and Qwen by 1/sqrt(128) after a norm: scores spread by about 1
    return r.normal(shape, kt, 2.0 if hk == 8 else 1.3), r.normal(shape, vt)


def _new(case, seed, layer):
    """What the program hands over for one layer."""
    hq, hk, d, _ = _dims(case)
    r = _Draws(seed, 2 * layer + 1)
    x = {}
    if case["kind"] == "block":
        n = 1024 if hk == 8 else 2048
        x["hidden"] = r.normal((n,), torch.float32 if hk == 8 else torch.float16)
        x["norm"] = 1 + r.normal((n,), std=0.1)
        sizes = (("q", hq * d, n), ("k", hk * d, n), ("v", hk * d, n), ("o", n, hq * d))
        for name, rows, cols in sizes:
            std = 2.0 / math.sqrt(cols)
            x[name] = r.q4(rows, cols, std) if case["weights"] == "q4" else r.normal((rows, cols), std=std)
        if hk == 4:
            x["post"] = 1 + r.normal((n,), std=0.1)
    else:
        s, t = case.get("sequences", 1), case.get("tokens", 1)
        wide = case["kind"] == "step" or case["kd"] == "f32" or (hk == 8 and case["kind"] == "decode")
        dt = torch.float32 if wide else DTYPES[case["kd"]][0]
        x["q"] = r.normal((s, t, hq, d), dt, 4.0 if hk == 8 else 1.0)
        x["k"] = r.normal((s, t, hk, d), dt, 2.0 if hk == 8 else 1.0)
        x["v"] = r.normal((s, t, hk, d), dt)
    if hk == 4:
        x["qn"], x["kn"] = 1.2 + r.normal((d,), std=0.1), 1.2 + r.normal((d,), std=0.1)
    return x


def _rows(arena, case, begin, count):
    """The cache's own memory of positions [begin, begin + count): keys, and values where they are not coded."""
    hq, hk, d, _ = _dims(case)
    y, desc, base = arena.layout, arena.desc, arena.arena.data_ptr()

    def part(address, dtype, positions):
        size = torch.tensor([], dtype=dtype).element_size()
        n = desc.layers * desc.sequences * hk * positions * d
        return arena.arena[address - base:address - base + n * size].view(dtype).view(
            desc.layers, desc.sequences, hk, positions, d)

    keys = part(y.keys, DTYPES[case["kd"]][0], desc.capacity)[:, :, :, begin:begin + count]
    if case["vd"] == "tiered":  # the window's slot of a single new row
        slot = begin % WINDOW
        return keys, part(y.value_ring, torch.float16, WINDOW)[:, :, :, slot:slot + 1]
    return keys, part(y.values, DTYPES[case["vd"]][0], desc.capacity)[:, :, :, begin:begin + count]


def prepare(case, seed):
    kind, ctx, layers = case["kind"], _context(), _layers(case)
    hq, hk, d, shape = _dims(case)
    tokens = case.get("tokens", 1)
    start = case["begin"] + case["count"] if kind == "leaves" else _start(case)
    end = start + (0 if kind == "leaves" else tokens)
    arena = rt.KvArena(ctx, shape, layers, case.get("sequences", 1), max(end, 1), DTYPES[case["kd"]][1],
                       DTYPES[case["vd"]][1], value_window=WINDOW if case["vd"] == "tiered" else 0)
    st = {"case": case, "arena": arena, "start": start, "layers": []}
    for layer in range(layers):
        if start:
            k, v = _past(case, seed, layer)
            if k.dtype != v.dtype:
                k, v = k.float(), v.float()
            with rt.Graph(ctx) as g:
                rt.store_kv(g, arena, layer, 0, k, v)
            del k, v
        if kind != "leaves":
            st["layers"].append(_new(case, seed, layer))
    if kind == "leaves":
        st["out"] = torch.empty((case["sequences"], case["count"], 32), dtype=torch.uint8, device=DEV)
        return st
    st["rows"] = _rows(arena, case, start, tokens)
    if kind == "block":
        _prepare_block(case, st)
    else:
        for x in st["layers"]:
            if kind == "step":
                for name in ("q", "k", "v"):
                    x[name] = x[name].view(-1, d)
            x["rot"] = torch.empty_like(x["q"])
            x["out"] = torch.empty_like(x["q"])
        if kind == "prompt":
            need = rt.prefill_workspace_bytes(arena, tokens)
        else:
            need = rt.attention_workspace_bytes(arena, case.get("sequences", 1), end)
        st["ws"] = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
    return st


def _prepare_block(case, st):
    arena, layers, end = st["arena"], st["layers"], st["start"] + 1
    granite, q4 = case["shape"] == "granite", case["weights"] == "q4"
    for x in layers:
        m = {}
        for name in ("q", "k", "v", "o"):
            if q4:
                codes, scales = x[name]
                m[name] = rt.Q4Matrix(codes, scales.view(torch.int16), codes.shape[0], 2 * codes.shape[1])
            else:
                m[name] = x[name]
        if not granite:
            x["w"] = rt.QwenQ4Layer(x["norm"], m["q"], m["k"], m["v"], x["qn"], x["kn"], m["o"], x["post"])
        else:
            x["w"] = (rt.GraniteQ4Layer if q4 else rt.GraniteLayer)(x["norm"], m["q"], m["k"], m["v"], m["o"])
    st["out"] = torch.stack([torch.empty_like(x["hidden"]) for x in layers])
    # the router norm's inverse of each Granite layer's result; Qwen's normalised one
    st["next"] = torch.empty(len(layers), device=DEV) if granite else torch.empty_like(st["out"])
    size = rt.granite_block_workspace_bytes if granite else rt.qwen_block_workspace_bytes
    st["ws"] = torch.empty(size(arena, end), dtype=torch.uint8, device=DEV)
    if case["replay"]:
        with torch.cuda.stream(torch.cuda.Stream()):  # a capture needs a stream of its own
            g = rt.Graph(_context())
            g.capture_begin()
            _encode_block(g, st)
            st["replay"] = g.capture_end()
            g.discard()


def _encode_block(g, st):
    case, arena, position = st["case"], st["arena"], st["start"]
    for i, x in enumerate(st["layers"]):
        if case["shape"] == "qwen":
            rt.qwen_attention_block(g, arena, i, position, x["w"], x["hidden"], st["out"][i], st["next"][i], st["ws"])
        elif case["weights"] == "q4":
            rt.granite_attention_block_q4(g, arena, i, position, x["w"], x["hidden"], st["out"][i], st["ws"],
                                          st["next"][i:i + 1])
        else:
            rt.granite_attention_block(g, arena, i, position, x["w"], x["hidden"], st["out"][i], st["ws"])


def run(st):
    case, arena, start = st["case"], st["arena"], st["start"]
    kind = case["kind"]
    if kind == "leaves":
        with rt.Graph(_context()) as g:
            arena.leaf_hashes(g, 0, case["begin"], case["count"], 0, case["sequences"], out=st["out"])
        return st["out"]
    if kind == "block":
        if case["replay"]:
            st["replay"].launch()
        else:
            arena.set_len(start)
            with rt.Graph(_context()) as g:
                _encode_block(g, st)
        more = [st["next"]] if case["weights"] == "q4" else []
        return {"hidden": st["out"], "next": more, "rows": st["rows"]}
    arena.set_len(start)
    with rt.Graph(_context()) as g:
        for i, x in enumerate(st["layers"]):
            if kind == "step":
                rt.decode_step(g, arena, i, start, x["q"], x["k"], x["v"], query_out=x["rot"], out=x["out"],
                               workspace=st["ws"])
                continue
            rt.rope_kv_batch(g, arena, i, start, x["q"], x["k"], x["v"], query_out=x["rot"],
                             query_norm=x.get("qn"), key_norm=x.get("kn"))
            if kind == "prompt":
                rt.prefill_attention(g, arena, i, start, x["rot"][0], out=x["out"][0], workspace=st["ws"])
            else:
                rt.attention(g, arena, i, x["rot"][:, 0], start + 1, out=x["out"][:, 0], workspace=st["ws"])
    return {"out": [x["out"] for x in st["layers"]], "rows": st["rows"]}


# ---- what a pass cannot do without -------------------------------------------------

def work(case):
    hq, hk, d, _ = _dims(case)
    row = hk * d * (BYTES[case["kd"]] + BYTES[case["vd"]])
    s, layers = case.get("sequences", 1), _layers(case)
    if case["kind"] == "leaves":
        return {"bytes": s * case["count"] * (row + 32), "flops": 0}
    t, start = case.get("tokens", 1), _start(case)
    pairs = s * t * (start + (t + 1) / 2)  # (query row, position) pairs
    flops = 4 * hq * d * pairs
    kv = s * (start + t) * row
    if case["vd"] == "tiered":
        kv += s * WINDOW * hk * d * (2 - BYTES["tiered"])
    if case["kind"] == "block":
        n = 1024 if hk == 8 else 2048
        cells = n * (hq + 2 * hk) * d + hq * d * n
        weight = 0.5 + 2 / 32 if case["weights"] == "q4" else 4
        return {"bytes": layers * (kv + cells * weight + 2 * n * (4 if hk == 8 else 2)),
                "flops": layers * (flops + 2 * cells)}
    size = 4 if case["kind"] == "step" or case["kd"] == "f32" or (hk == 8 and case["kind"] == "decode") else 2
    return {"bytes": layers * (kv + s * t * (2 * hq + 2 * hk) * d * size), "flops": layers * flops}


def tolerance(case):
    if case["kind"] == "leaves":
        return "exact"
    # about four times what the path is off the 64-bit result
    if case["kd"] == "f32":
        # 32-bit products and sums; a new value row is rounded once to a 16-bit cache, where a tie may fall either way
        return {"rel": 1e-5, "max": 1e-3}
    if case["kd"] == "f16":  # 16-bit rows, probabilities and results
        return {"rel": 1.5e-3}
    return {"rel": 7e-3}


# ---- the same in 64 bits -------------------------------------------------------------

def _rope(x, positions, theta):
    """Rotate-half of x [..., T, heads, d] in float64; the angle is a binary32 product, as the models define it."""
    d = x.shape[-1]
    freq = (np.float64(theta) ** (-np.arange(d // 2) / (d // 2))).astype(np.float32)
    angle = (positions.float()[:, None] * torch.from_numpy(freq).to(DEV)).double()[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    c, s = torch.cos(angle), torch.sin(angle)
    return torch.cat((a * c - b * s, a * s + b * c), -1)


def _rms(x, weight):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-6) * weight.double()


def _front(case, x, q, k):
    """q [S][T][Hq][d], k [S][T][Hkv][d] in float64: per-head norm (Qwen), then RoPE at the new positions."""
    qwen = _dims(case)[1] == 4
    positions = torch.arange(_start(case), _start(case) + q.shape[1], device=DEV)
    if qwen:
        q, k = _rms(q, x["qn"]), _rms(k, x["kn"])
    theta = 1e6 if qwen else 1e4
    return _rope(q, positions, theta), _rope(k, positions, theta)


def _as_stored(x, dtype):
    return x.to(dtype).double()


def _coded(v):
    """Value rows as the INT8 tier holds them: one binary16 scale per 32 elements."""
    b = v.view(*v.shape[:-1], -1, 32)
    scale = (b.abs().amax(-1, keepdim=True).float() / 127).to(torch.float16).double()
    code = torch.where(scale > 0, (b / scale).float().round().clamp(-127, 127).double(), torch.zeros_like(b))
    return (code * scale).view_as(v)


def _attend(case, q, k, v):
    """q [S][T][Hq][d] over k, v [S][L][Hkv][d], all float64; the T rows are the last T positions."""
    s, t, hq, d = q.shape
    length, hk = k.shape[1], k.shape[2]
    scale = 1 / 64 if hk == 8 else 1 / math.sqrt(d)
    out = torch.empty_like(q)
    block = max(1, min(t, (1 << 27) // length))
    for i in range(s):
        for h in range(hk):
            kt, vh = k[i, :, h].t().contiguous(), v[i, :, h].contiguous()
            heads = slice(h * (hq // hk), (h + 1) * (hq // hk))
            qh = q[i, :, heads]
            for a in range(0, t, block):
                part = qh[a:a + block]
                w = part.reshape(-1, d) @ kt * scale
                w = w.view(part.shape[0], -1, length)
                if t > 1:
                    seen = torch.arange(a, a + part.shape[0], device=DEV)[:, None] + (length - t)
                    w.masked_fill_((torch.arange(length, device=DEV)[None] > seen)[:, None], -math.inf)
                w = torch.softmax(w, -1)
                out[i, a:a + block, heads] = (w.view(-1, length) @ vh).view_as(part)
    return out


def _weight(w):
    if not isinstance(w, tuple):
        return w.double()
    codes, scales = w
    both = torch.stack((codes & 15, codes >> 4), -1).view(codes.shape[0], -1).double() - 7
    return (both.view(codes.shape[0], -1, 32) * scales.double()[..., None]).view(codes.shape[0], -1)


def exact(case, seed):
    if case["kind"] == "leaves":
        return None
    hq, hk, d, _ = _dims(case)
    kt, vt = DTYPES[case["kd"]][0], DTYPES[case["vd"]][0]
    out, after, keys, values = [], [], [], []
    for layer in range(_layers(case)):
        x = _new(case, seed, layer)
        if case["kind"] == "block":
            hidden = x["hidden"].double()
            n = _rms(hidden, x["norm"])
            q, k, v = ((_weight(x[name]) @ n).view(1, 1, -1, d) for name in ("q", "k", "v"))
        else:
            q, k, v = (x[name].double() for name in ("q", "k", "v"))
        q, k = _front(case, x, q, k)
        if case["kind"] != "block":
            q = _as_stored(q, x["q"].dtype)  # the program's own buffer for the rotated query
        k, v = _as_stored(k, kt), _as_stored(v, vt)
        keys.append(k.transpose(1, 2))
        values.append(v.transpose(1, 2))
        pk, pv = (p.double() for p in _past(case, seed, layer)) if _start(case) else (k[:, :0], v[:, :0])
        if case["vd"] == "tiered":
            old = max(0, _start(case) + 1 - WINDOW)
            pv[:, :old] = _coded(pv[:, :old].contiguous())
        att = _attend(case, q, torch.cat((pk, k), 1), torch.cat((pv, v), 1))
        del pk, pv
        if case["kind"] == "step":
            att = att.view(hq, d)
        if case["kind"] != "block":
            out.append(att)
            continue
        o = _weight(x["o"]) @ att.reshape(-1)
        if hk == 8:
            out.append(hidden + float(np.float32(0.22)) * o)
            after.append(1 / torch.sqrt(out[-1].square().mean() + 1e-6))
        else:
            out.append(_as_stored(hidden + o, torch.float16))
            after.append(_rms(out[-1], x["post"]))
    rows = (torch.stack(keys), torch.stack(values))
    if case["kind"] != "block":
        return {"out": out, "rows": rows}
    more = [torch.stack(after)] if case["weights"] == "q4" else []
    return {"hidden": torch.stack(out), "next": more, "rows": rows}

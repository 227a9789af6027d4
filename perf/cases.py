"""Performance cases: the work this framework does for a program, through its
public Python entry points (hotarubi_amd).

Every case is a plain dict; `kind` names the path, the other values its
sizes, formats and options:

  linear      one linear layer, or a stack of same-shaped layers in one
              launch: MXFP4 or W8 weights, MXINT8 or MXFP8 activations, fast
              or exact mode, DDR words, weight panels or W8 panels
  gated_mlp   RMSNorm + quantize, the gated pair (up; gate with SiLU and the
              product, requantized), down with the residual add
  gelu_mlp    LayerNorm + quantize, W8 up with GELU and requantize, W8 down
  bottleneck  a ResNet bottleneck's three convolutions as im2col GEMMs
  attention   SPLIT8 of K, T32_SPLIT8 of V, scores per head, softmax +
              quantize, the weighted values per head, in one HIP graph
  gacc        the deformable aggregation: 6 chained gather-accumulates
  encode      fp32 activations to MXINT8 / MXFP8 words

`exact` restates each path in float64 with plain torch from the same seeded
inputs.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import hotarubi_amd as hb

DEV = "cuda"
LOG2E = 1.4426950216293335  # the FP32 constant of the softmax program
EPS = 1e-6
GACC_POOL, GACC_CAMERAS, GACC_MAP = 100000, 6, 176  # feature rows; cameras; rows per map line


def listed():
    return [
        # the smallest call: one token through SmolVLA's up projection
        dict(name="decode_m1", kind="linear", m=1, k=960, n=2560, fmt="mxfp4", mode="fast",
             layout="panels", act="int8", layers=1, epilogue="none"),
        # the action expert's MLP on one chunk of 50 action tokens (latency)
        dict(name="expert_mlp_b1", kind="gated_mlp", m=50, width=736, hidden=2048, mode="fast"),
        # a decoder layer's MLP over the prefix of 32 requests of 141 tokens
        dict(name="prefix_mlp_b32", kind="gated_mlp", m=4512, width=960, hidden=2560,
             mode="fast"),
        # weights streamed from HBM: 256 layers of 128 rows in one launch
        dict(name="stack_mxfp4_m128", kind="linear", m=128, k=2560, n=960, fmt="mxfp4",
             mode="fast", layout="panels", act="int8", layers=256, epilogue="none"),
        # the same with FP8 activations at decode's 16 rows
        dict(name="stack_mxfp8_m16", kind="linear", m=16, k=2560, n=960, fmt="mxfp4",
             mode="fast", layout="panels", act="fp8", layers=256, epilogue="none"),
        # the vision encoder's MLP: two cameras of 1,024 patches, W8 weights
        dict(name="siglip_mlp_w8", kind="gelu_mlp", m=2048, width=768, hidden=3072, mode="fast",
             layout="w8_panels"),
        # the vision encoder's QKV, bit for bit the NPU's (the default mode)
        dict(name="siglip_qkv_exact", kind="linear", m=2048, k=768, n=2304, fmt="w8",
             mode="exact", layout="words", act="int8", layers=1, epilogue="scale_bias"),
        # a decoder layer's down projection over 32 requests, bit for bit
        dict(name="prefix_down_exact", kind="linear", m=4512, k=2560, n=960, fmt="mxfp4",
             mode="exact", layout="words", act="int8", layers=1, epilogue="residual"),
        # SparseDrive-S backbone, stage 1, one frame of 6 cameras (64 x 176)
        dict(name="bottleneck_f1", kind="bottleneck", positions=67584, mid=64),
        # the action expert's attention over 32 requests
        dict(name="attention_b32", kind="attention", batch=32, rows=50, prefix=128, suffix=64),
        # SparseDrive-S head, 4 frames: 900 anchors, 13 points on 4 levels
        dict(name="aggregate_f4", kind="gacc", quads=900, slots=52, blocks=8),
        # a model's input: the prefix embeddings of 32 requests
        dict(name="encode_prefix", kind="encode", rows=4512, cols=960, act="int8"),
    ]


def _log(rng, lo, hi, step=1):
    """An integer multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi // step * step, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "gated_mlp", "gelu_mlp", "bottleneck",
                       "attention", "gacc", "encode"])
    if kind == "linear":
        mode = rng.choice(["fast", "fast", "exact"])
        fmt = rng.choice(["mxfp4", "w8"])
        layout = rng.choice(["words", "panels"] + (["w8_panels"] if (fmt, mode) == ("w8", "fast")
                                                   else []))
        act = rng.choice(["int8", "fp8"]) if (fmt, mode, layout) == ("mxfp4", "fast", "panels") \
            else "int8"
        epilogue = rng.choice(["none", "scale_bias", "residual", "relu_q"])
        m, k, n = _log(rng, 1, 4512), _log(rng, 96, 2560, 32), _log(rng, 64, 2560, 32)
        # at most the work of the listed stack (fast) or down projection (exact)
        cap = 256 * 128 * 2560 * 960 if mode == "fast" else 4512 * 2560 * 960
        most = cap // (m * k * n * (2 if fmt == "w8" else 1))
        if most < 1:
            m, most = max(1, m // 4), 1
        layers = rng.choice([1, 1, _log(rng, 1, max(1, min(256, most)))])
        return dict(kind=kind, m=m, k=k, n=n, fmt=fmt, mode=mode, layout=layout, act=act,
                    layers=layers, epilogue=epilogue)
    if kind == "gated_mlp":
        return dict(kind=kind, m=_log(rng, 1, 4512), width=_log(rng, 256, 960, 32),
                    hidden=_log(rng, 512, 2560, 32), mode=rng.choice(["fast", "fast", "exact"]))
    if kind == "gelu_mlp":
        return dict(kind=kind, m=_log(rng, 16, 2048), width=_log(rng, 256, 768, 32),
                    hidden=_log(rng, 512, 3072, 32), mode="fast",
                    layout=rng.choice(["words", "panels", "w8_panels"]))
    if kind == "bottleneck":
        mid = rng.choice([64, 96, 128, 256])
        return dict(kind=kind, positions=_log(rng, 1056, 67584 * 64 // mid, 4), mid=mid)
    if kind == "attention":
        return dict(kind=kind, batch=_log(rng, 2, 32), rows=rng.randrange(17, 65),
                    prefix=rng.choice([64, 96, 128]), suffix=rng.choice([32, 64]))
    if kind == "gacc":
        return dict(kind=kind, quads=_log(rng, 25, 900), slots=rng.randrange(4, 53),
                    blocks=rng.choice([1, 2, 4, 8]))
    return dict(kind="encode", rows=_log(rng, 1, 4512), cols=_log(rng, 30, 2560),
                act=rng.choice(["int8", "fp8"]))


# ---------------------------------------------------------------- inputs --

def _rng(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _block_exponent(x, bias):
    """floor(log2 max|x|) - bias per 32 values (0 for a zero block)."""
    amax = x.abs().amax(-1)
    e = torch.frexp(amax)[1] - 1 - bias
    return torch.where(amax > 0, e, torch.zeros_like(e)).clamp(-127, 127)


def _words(codes, scale_bytes, pad_quads=True):
    """Codes [rows][kb][32] (uint8) and scale bytes [rows][kb] -> MXINT8 DDR
    words [ceil(rows/4) * kb][144]; rows past the end encode zeros."""
    rows, kb, _ = codes.shape
    quads = (rows + 3) // 4
    out = torch.zeros((quads, kb, 144), dtype=torch.uint8, device=DEV)
    c = torch.zeros((quads * 4, kb, 32), dtype=torch.uint8, device=DEV)
    s = torch.full((quads * 4, kb), 127, dtype=torch.uint8, device=DEV)
    c[:rows], s[:rows] = codes, scale_bytes
    out[:, :, :128] = c.view(quads, 4, kb, 32).transpose(1, 2).reshape(quads, kb, 128)
    out[:, :, 128:132] = s.view(quads, 4, kb).transpose(1, 2)
    return out.view(-1, 144)


def _quantize(x):
    """MXINT8 of x [rows][cols] (cols a multiple of 32): codes [rows][kb][32]
    as float64 and exponents [rows][kb]."""
    b = x.double().view(x.shape[0], -1, 32)
    e = _block_exponent(b, 0)
    q = torch.round(b * torch.exp2((6 - e).double()).unsqueeze(-1)).clamp(-128, 127)
    return q, e


def _mxint8(x):
    q, e = _quantize(x)
    return _words(q.to(torch.int8).view(torch.uint8), (e + 127).to(torch.uint8))


def _mxfp8(x):
    b = x.view(x.shape[0], -1, 32)
    e = _block_exponent(b, 8)
    y = (b * torch.exp2(-e.float()).unsqueeze(-1)).clamp(-448, 448)
    return _words(y.to(torch.float8_e4m3fn).view(torch.uint8), (e + 127).to(torch.uint8))


def _read_words(words, rows, kb, fp8=False):
    """The float64 values [rows][kb * 32] of activation words."""
    w = words.view(-1, kb, 144)
    codes = w[:, :, :128].reshape(-1, kb, 4, 32).transpose(1, 2).reshape(-1, kb, 32)
    e = w[:, :, 128:132].transpose(1, 2).reshape(-1, kb).double() - (127 if fp8 else 133)
    v = codes.contiguous().view(torch.float8_e4m3fn if fp8 else torch.int8).double()
    return (v * torch.exp2(e).unsqueeze(-1)).reshape(-1, kb * 32)[:rows]


def _weights(g, n, kb, w8):
    """Weight words of a layer: one MXFP4 plane (random E2M1 codes, exponents
    -10..-2) or the two nibble planes of random int8 weights."""
    planes = []
    for _ in range(2 if w8 else 1):
        w = torch.randint(0, 256, (n // 8 * kb, 144), generator=g, device=DEV, dtype=torch.uint8)
        w[:, 136:] = 0
        if w8:
            w[:, 128:136] = 133
        else:
            w[:, 128:136] = torch.randint(117, 126, (n // 8 * kb, 8), generator=g, device=DEV,
                                          dtype=torch.uint8)
        planes.append(w)
    return planes


def _read_weights(planes, n, kb):
    """The float64 weights [n][kb * 32] of a layer's DDR words."""
    total = 0
    e2m1 = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12],
                        dtype=torch.float64, device=DEV)
    hi = torch.tensor([v if v < 8 else v - 16 for v in range(16)], dtype=torch.float64, device=DEV)
    lo = torch.arange(16, dtype=torch.float64, device=DEV)
    for i, p in enumerate(planes):
        table, bias = (e2m1, -7) if len(planes) == 1 else ((hi, -8) if i == 0 else (lo, -12))
        w = p.view(n // 8, kb, 144)
        b = w[:, :, :128].reshape(n // 8, kb, 8, 16)
        nib = torch.stack((b & 15, b >> 4), -1).reshape(n // 8, kb, 8, 32).long()
        # (an activation's scale is 2^(ea-133); the weight's share of the
        # block value 2^(ea + ew + bias - 254) is 2^(ew + bias - 121))
        e = w[:, :, 128:136].double() + bias - 121
        v = table[nib] * torch.exp2(e).unsqueeze(-1)
        total = total + v.permute(0, 2, 1, 3).reshape(n, kb * 32)
    return total


def _pack(planes, n, kb, layout):
    """The planes in the layout a program keeps them in, packed once."""
    if layout == "words":
        return planes
    if layout == "w8_panels":
        out = torch.empty(hb.w8_panel_bytes(n, kb), dtype=torch.uint8, device=DEV)
        hb.pack_w8(planes[0], planes[1], n, kb, out, ctx=_ctx())
        return [out, out]
    packed = []
    for p in planes:
        out = torch.empty(hb.panel_bytes(n, kb), dtype=torch.uint8, device=DEV)
        hb.pack_weights(p, n, kb, out, ctx=_ctx())
        packed.append(out)
    return packed


def _table(kind):
    """TBUF: [0, 512) 2^(i/512), [512, 1024) the activation at i/32; value
    and slope as FP32."""
    i = np.arange(513, dtype=np.float64)
    x = i / 32.0
    act = 1.0 / (1.0 + np.exp(-x)) if kind == "silu" else \
        0.5 * (1.0 + np.tanh(np.sqrt(2.0 / np.pi) * (x + 0.044715 * x ** 3)))
    out = np.zeros(1024, np.uint64)
    for base, v in ((0, np.exp2(i / 512)), (512, act)):
        vb = v.astype(np.float32)
        slope = (vb[1:].astype(np.float64) - vb[:-1]).astype(np.float32)
        out[base:base + 512] = (slope.view(np.uint32).astype(np.uint64) << np.uint64(32)) | \
            vb[:-1].view(np.uint32).astype(np.uint64)
    return out


def _table_on_gpu(kind):
    return torch.from_numpy(_table(kind).view(np.int64)).to(DEV)


_contexts = {}


def _ctx(graph=False):
    """The program's context, on torch's current stream (or, for a path that
    is captured once, on the stream it is captured on)."""
    if graph not in _contexts:
        ctx = hb.Context(torch.cuda.current_device())
        stream = torch.cuda.Stream() if graph else torch.cuda.current_stream()
        ctx.set_stream(stream.cuda_stream)
        _contexts[graph] = (ctx, stream)
    return _contexts[graph][0]


def _f32_bits(v):
    return int(np.array(v, np.float32).view(np.uint32))


def _mode(name):
    return hb.FAST if name == "fast" else hb.EXACT


def _inputs(case, seed):
    """The seeded inputs of a case, as plain tensors: what both `prepare` and
    `exact` start from."""
    g, kind, s = _rng(seed), case["kind"], {}
    if kind == "linear":
        m, kb, n, layers, w8 = case["m"], case["k"] // 32, case["n"], case["layers"], \
            case["fmt"] == "w8"
        enc = _mxfp8 if case["act"] == "fp8" else _mxint8
        s["a"] = [enc(_randn(g, m, kb * 32)) for _ in range(layers)]
        s["w"] = [_weights(g, n, kb, w8) for _ in range(layers)]
        s["scale"] = torch.rand((layers, n), generator=g, device=DEV) * 0.019 + 0.001
        s["bias"] = _randn(g, layers, n) * 0.1
        if case["epilogue"] == "residual":
            s["x"] = _randn(g, layers, m, n)
    elif kind in ("gated_mlp", "gelu_mlp"):
        m, d, h = case["m"], case["width"], case["hidden"]
        s["x"] = _randn(g, m, d)
        s["gamma"] = torch.rand((d,), generator=g, device=DEV) + 0.5
        s["beta"] = _randn(g, d) * 0.1
        w8 = kind == "gelu_mlp"
        s["w_up"] = _weights(g, h, d // 32, w8)
        if not w8:
            s["w_gate"] = _weights(g, h, d // 32, w8)
        s["w_down"] = _weights(g, d, h // 32, w8)
        for name, size in (("up", h), ("down", d)):
            s["s_" + name] = torch.rand((size,), generator=g, device=DEV) * 0.0002 + 0.0003
            s["b_" + name] = _randn(g, size) * 0.1
    elif kind == "bottleneck":
        p, mid = case["positions"], case["mid"]
        cout = 4 * mid
        s["x"] = _mxint8(_randn(g, p, cout).relu_())
        s["cols"] = _mxint8(_randn(g, p, 9 * mid).relu_())  # the 3x3 im2col words
        s["residual"] = _randn(g, p, cout).relu_()
        s["w1"] = _weights(g, mid, cout // 32, False)
        s["w2"] = _weights(g, mid, 9 * mid // 32, False)
        s["w3"] = _weights(g, cout, mid // 32, False)
        s["b1"], s["b2"], s["b3"] = _randn(g, mid) * 0.1, _randn(g, mid) * 0.1, \
            _randn(g, cout) * 0.1
    elif kind == "attention":
        b, rows, keys = case["batch"], case["rows"], case["prefix"] + case["suffix"]
        pad = (rows + 3) // 4 * 4
        s["q"] = _mxint8(_randn(g, b * pad, 960)).view(b, -1, 144)
        s["k"] = _mxint8(_randn(g, b * keys, 320))
        s["v"] = _mxint8(_randn(g, b * keys, 320))
        mask = torch.zeros((rows, keys), device=DEV)
        mask[:, case["prefix"]:] = -1e4 * torch.triu(torch.ones(rows, case["suffix"], device=DEV), 1)
        s["mask"] = mask
    elif kind == "gacc":
        s = _gacc_inputs(case, g)
    else:
        s["x"] = _randn(g, case["rows"], case["cols"])
    return s


def _gacc_inputs(case, g):
    """One image: the feature rows (MXINT8 row format), the weights of every
    quad, and per camera the lists; a point's 4 entries are the corners of a
    map cell, a tenth of the points lie outside the camera (null)."""
    quads, slots, blocks = case["quads"], case["slots"], case["blocks"]
    size = hb.row_token_bytes(blocks)
    w_words = (slots + 7) // 8
    w_bytes, list_bytes = blocks * w_words * 128, 16 + 128 * slots
    pool = torch.randint(0, 256, (GACC_POOL, size), generator=g, device=DEV, dtype=torch.uint8)
    pool[:, 32 * blocks:33 * blocks] = torch.randint(118, 127, (GACC_POOL, blocks), generator=g,
                                                     device=DEV, dtype=torch.uint8)
    w = torch.rand((quads, blocks, w_words, 4, 8), generator=g, device=DEV) * 0.04
    cells = torch.randint(0, GACC_POOL - GACC_MAP - 1, (GACC_CAMERAS, quads, slots, 4, 1),
                          generator=g, device=DEV)
    corner = torch.tensor([0, 1, GACC_MAP, GACC_MAP + 1], device=DEV)
    rows = cells + corner  # [camera][quad][slot][token][point]
    out = torch.rand((GACC_CAMERAS, quads, slots, 4, 1), generator=g, device=DEV) < 0.1
    f = torch.rand((2, GACC_CAMERAS, quads, slots, 4), generator=g, device=DEV)
    bw = torch.stack(((1 - f[0]) * (1 - f[1]), f[0] * (1 - f[1]), (1 - f[0]) * f[1], f[0] * f[1]), -1)
    w_base = GACC_POOL * size
    list_base = w_base + quads * w_bytes
    entry = torch.where(out, torch.full_like(rows, 0xFFFFFFFF), rows * (size // 16))
    entry = entry | (bw.contiguous().view(torch.int32).long() << 32)
    lists = torch.zeros((GACC_CAMERAS, quads, list_bytes), dtype=torch.uint8, device=DEV)
    head = (w_base + torch.arange(quads, device=DEV) * w_bytes) // 16
    lists[:, :, :8] = head.view(-1, 1).view(torch.uint8)
    lists[:, :, 16:] = entry.contiguous().view(GACC_CAMERAS, quads, slots * 16).view(torch.uint8)
    img = torch.cat((pool.view(-1), w.view(-1).view(torch.uint8), lists.view(-1)))
    return dict(img=img, list_base=list_base, list_bytes=list_bytes, w_stride=w_words * 8,
                pool=pool, w=w, rows=rows, out=out.expand_as(rows), bw=bw)


# --------------------------------------------------------------- prepare --

def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    s["kind"] = kind
    build = globals()["_prepare_" + kind]
    build(case, s)
    torch.cuda.synchronize()
    return s


def _ops(case, s, i):
    e = case["epilogue"]
    if e == "scale_bias":
        return [(hb.EP_MULP, s["scale"][i]), (hb.EP_ADDP, s["bias"][i])]
    if e == "residual":
        return [(hb.EP_ADD, s["x"][i])]
    if e == "relu_q":
        return [(hb.EP_ADDP, s["bias"][i]), (hb.EP_RELU, None)]
    return []


def _prepare_linear(case, s):
    m, kb, n, layers = case["m"], case["k"] // 32, case["n"], case["layers"]
    lay, w8 = case["layout"], case["fmt"] == "w8"
    a = torch.stack(s["a"])
    packed = [_pack(p, n, kb, lay) for p in s["w"]]
    w = [torch.stack([p[l] for p in packed]) for l in range(1 if lay == "w8_panels" or not w8 else 2)]
    if lay == "w8_panels":
        w = [w[0], w[0]]
    c = torch.empty((layers, m, n), device=DEV)
    quant = case["epilogue"] == "relu_q"
    q = torch.zeros((layers, (m + 3) // 4 * (n // 32), 144), dtype=torch.uint8, device=DEV) \
        if quant else None
    s.update(a=a, w=w, c=c, q=q)
    s["descs"] = [hb.linear_desc(m, n, kb, a[i], [p[i] for p in w], [1, 2] if w8 else [0], c[i],
                                 ops=_ops(case, s, i), mode=_mode(case["mode"]),
                                 q_out=q[i] if quant else None, panels=lay == "panels",
                                 w8_panels=lay == "w8_panels", a_fp8=case["act"] == "fp8")
                  for i in range(layers)]


def _prepare_gated_mlp(case, s):
    m, d, h = case["m"], case["width"], case["hidden"]
    quads, mode = (m + 3) // 4, _mode(case["mode"])
    s.update(dims=(m, d), table=_table_on_gpu("silu"), gated=True,
             normed=torch.empty((quads * (d // 32), 144), dtype=torch.uint8, device=DEV),
             up=torch.empty((m, h), device=DEV), gate=torch.empty((m, h), device=DEV),
             hid=torch.empty((quads * (h // 32), 144), dtype=torch.uint8, device=DEV),
             y=torch.empty((m, d), device=DEV))
    for name in ("w_up", "w_gate"):
        s[name] = _pack(s[name], h, d // 32, "panels")
    s["w_down"] = _pack(s["w_down"], d, h // 32, "panels")
    up = hb.linear_desc(m, h, d // 32, s["normed"], s["w_up"], [0], s["up"], mode=mode, panels=True)
    gate = hb.linear_desc(m, h, d // 32, s["normed"], s["w_gate"], [0], s["gate"], mode=mode,
                          panels=True, ops=[(hb.EP_ACT_MUL, s["up"])], tbuf=s["table"],
                          q_out=s["hid"])
    s["down"] = hb.linear_desc(m, d, h // 32, s["hid"], s["w_down"], [0], s["y"], mode=mode,
                               panels=True, ops=[(hb.EP_ADD, s["x"])])
    s["pair"] = (type(up) * 2)(up, gate)


def _prepare_gelu_mlp(case, s):
    m, d, h, lay = case["m"], case["width"], case["hidden"], case["layout"]
    quads, mode = (m + 3) // 4, _mode(case["mode"])
    kinds = dict(panels=lay == "panels", w8_panels=lay == "w8_panels", mode=mode)
    s.update(dims=(m, d), table=_table_on_gpu("gelu"), gated=False,
             normed=torch.empty((quads * (d // 32), 144), dtype=torch.uint8, device=DEV),
             up=torch.empty((m, h), device=DEV),
             hid=torch.empty((quads * (h // 32), 144), dtype=torch.uint8, device=DEV),
             y=torch.empty((m, d), device=DEV))
    s["w_up"] = _pack(s["w_up"], h, d // 32, lay)
    s["w_down"] = _pack(s["w_down"], d, h // 32, lay)
    s["first"] = hb.linear_desc(
        m, h, d // 32, s["normed"], s["w_up"], [1, 2], s["up"], tbuf=s["table"], q_out=s["hid"],
        ops=[(hb.EP_MULP, s["s_up"]), (hb.EP_ADDP, s["b_up"]), (hb.EP_ACT, None)], **kinds)
    s["down"] = hb.linear_desc(
        m, d, h // 32, s["hid"], s["w_down"], [1, 2], s["y"],
        ops=[(hb.EP_MULP, s["s_down"]), (hb.EP_ADDP, s["b_down"])], **kinds)


def _prepare_bottleneck(case, s):
    p, mid = case["positions"], case["mid"]
    cout, quads = 4 * mid, (p + 3) // 4

    def words(n):
        return torch.empty((quads * (n // 32), 144), dtype=torch.uint8, device=DEV)

    s.update(t1=words(mid), t2=words(mid), y8=words(cout), y=torch.empty((p, cout), device=DEV))
    for name, n, kb in (("w1", mid, cout // 32), ("w2", mid, 9 * mid // 32), ("w3", cout, mid // 32)):
        s[name] = _pack(s[name], n, kb, "panels")
    relu = (hb.EP_RELU, None)
    s["descs"] = [
        hb.linear_desc(p, mid, cout // 32, s["x"], s["w1"], [0], None, q_out=s["t1"], mode=hb.FAST,
                       panels=True, ops=[(hb.EP_ADDP, s["b1"]), relu]),
        hb.linear_desc(p, mid, 9 * mid // 32, s["cols"], s["w2"], [0], None, q_out=s["t2"],
                       mode=hb.FAST, panels=True, ops=[(hb.EP_ADDP, s["b2"]), relu]),
        hb.linear_desc(p, cout, mid // 32, s["t2"], s["w3"], [0], s["y"], q_out=s["y8"],
                       mode=hb.FAST, panels=True,
                       ops=[(hb.EP_ADDP, s["b3"]), (hb.EP_ADD, s["residual"]), relu])]


def _prepare_attention(case, s):
    """15 query heads over 5 KV heads of 64, `rows` queries per element."""
    b, rows, keys = case["batch"], case["rows"], case["prefix"] + case["suffix"]
    heads, kvw, qw, quads, kbk = 15, 10, 30, (rows + 3) // 4, keys // 32
    s["kh"] = torch.empty((2, b * keys // 8 * kvw, 144), dtype=torch.uint8, device=DEV)
    s["vh"] = torch.empty((2, 4 * kvw * b * kbk, 144), dtype=torch.uint8, device=DEV)
    s["scores"] = torch.zeros((b, heads, quads * 4, keys), device=DEV)
    s["p"] = torch.zeros((b * heads, quads * kbk, 144), dtype=torch.uint8, device=DEV)
    s["o"] = torch.empty((b, heads, rows, 64), device=DEV)
    s["table"] = _table_on_gpu("silu")
    ops = [(hb.EP_ADD, s["mask"]), (hb.EP_SCALE, _f32_bits(0.125))]
    qk, pv = [], []
    for h in range(heads):
        j = h // 3
        qk.append([hb.linear_desc(rows, keys, kvw, s["q"][e, 2 * h:],
                                  [s["kh"][l, e * keys // 8 * kvw + 2 * j:] for l in range(2)],
                                  [1, 2], s["scores"][e, h], pieces=[(0, 2, 0)], a_stride=qw,
                                  ops=ops, mode=hb.FAST) for e in range(b)])
        pv.append([hb.linear_desc(rows, 64, b * kbk, s["p"][e * heads + h],
                                  [s["vh"][l, 8 * j * b * kbk + e * kbk:] for l in range(2)],
                                  [1, 2], s["o"][e, h], pieces=[(0, kbk, 0)], a_stride=kbk,
                                  mode=hb.FAST) for e in range(b)])

    def step(ctx):
        hb.split8(s["k"], b * keys // 4, kvw, s["kh"][0], s["kh"][1], ctx=ctx, sync=False)
        hb.t32_split8(s["v"], b * keys // 4, kvw, s["vh"][0], s["vh"][1], ctx=ctx, sync=False)
        for group in qk:
            hb.linear_batched(group, ctx)
        hb.rows(hb.ROWS_SOFTMAX, s["scores"], b * heads * quads * 4, keys, keys, tbuf=s["table"],
                q_out=s["p"], ctx=ctx, sync=False)
        for group in pv:
            hb.linear_batched(group, ctx)

    ctx = _ctx(graph=True)
    stream = _contexts[True][1]
    stream.wait_stream(torch.cuda.current_stream())
    step(ctx)
    stream.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"], stream=stream):
        step(ctx)


def _prepare_gacc(case, s):
    for name in ("pool", "w", "rows", "out", "bw"):
        del s[name]
    s["acc"] = torch.empty((case["quads"] * 4, 32 * case["blocks"]), device=DEV)
    s["case"] = dict(case)
    s["lists"] = [s["img"][s["list_base"] + c * case["quads"] * s["list_bytes"]:]
                  for c in range(GACC_CAMERAS)]


def _prepare_encode(case, s):
    s["case"] = dict(case)
    s["words"] = torch.empty(((case["rows"] + 3) // 4 * ((case["cols"] + 31) // 32), 144),
                             dtype=torch.uint8, device=DEV)


# ------------------------------------------------------------------- run --

def run(s):
    kind, ctx = s["kind"], _ctx()
    if kind == "linear":
        if len(s["descs"]) == 1:
            hb.launch(s["descs"][0], ctx)
        else:
            hb.linear_batched(s["descs"], ctx)
        return {"c": s["c"], "q": s["q"]}
    if kind in ("gated_mlp", "gelu_mlp"):
        m, d = s["dims"]
        entry = hb.ROWS_RMSNORM if s["gated"] else hb.ROWS_LAYERNORM
        hb.rows(entry, s["x"], m, d, d, _f32_bits(EPS), s["gamma"],
                None if s["gated"] else s["beta"], q_out=s["normed"], ctx=ctx, sync=False)
        if s["gated"]:
            hb.linear_group(s["pair"], ctx)
        else:
            hb.launch(s["first"], ctx)
        hb.launch(s["down"], ctx)
        return {"normed": s["normed"], "up": s["up"], "hid": s["hid"], "y": s["y"]}
    if kind == "bottleneck":
        for d in s["descs"]:
            hb.launch(d, ctx)
        return {"t1": s["t1"], "t2": s["t2"], "y": s["y"], "y8": s["y8"]}
    if kind == "attention":
        s["graph"].replay()
        return {"scores": s["scores"], "p": s["p"], "o": s["o"]}
    if kind == "gacc":
        c = s["case"]
        for i, lst in enumerate(s["lists"]):
            hb.gacc(s["img"], lst, c["quads"], c["slots"], c["blocks"], s["w_stride"], s["acc"],
                    list_stride=s["list_bytes"], accumulate=i > 0, ctx=ctx, sync=False)
        return s["acc"]
    c = s["case"]
    (hb.encode_mxfp8 if c["act"] == "fp8" else hb.encode_mxint8)(
        s["x"], c["rows"], c["cols"], s["words"], ctx=ctx)
    return s["words"]


# ------------------------------------------------------------------ work --

def _layer_bytes(m, k, n, w8, c=True, q=False, layers=1):
    """A (MXINT8), W, the FP32 output and the requantized words."""
    return layers * (m * k * 33 / 32 + n * k * ((1 if w8 else 0.5) + 1 / 32)
                     + (4 * m * n if c else 0) + (m * n * 33 / 32 if q else 0))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n, layers = case["m"], case["k"], case["n"], case["layers"]
        nbytes = _layer_bytes(m, k, n, case["fmt"] == "w8", q=case["epilogue"] == "relu_q",
                              layers=layers)
        nbytes += layers * {"none": 0, "scale_bias": 8 * n, "residual": 4 * m * n,
                            "relu_q": 4 * n}[case["epilogue"]]
        return {"bytes": nbytes, "flops": 2 * m * k * n * layers}
    if kind in ("gated_mlp", "gelu_mlp"):
        m, d, h, w8 = case["m"], case["width"], case["hidden"], kind == "gelu_mlp"
        ups = 1 if w8 else 2
        # the rows and their normed words; up (and gate) with FP32 and words
        # out; down with the residual
        nbytes = m * d * 4 + m * d * 33 / 32 + ups * _layer_bytes(m, d, h, w8) + m * h * 33 / 32
        nbytes += _layer_bytes(m, h, d, w8) + (0 if w8 else 4 * m * d)
        return {"bytes": nbytes, "flops": 2 * m * d * h * (ups + 1)}
    if kind == "bottleneck":
        p, mid = case["positions"], case["mid"]
        nbytes = _layer_bytes(p, 4 * mid, mid, False, c=False, q=True) \
            + _layer_bytes(p, 9 * mid, mid, False, c=False, q=True) \
            + _layer_bytes(p, mid, 4 * mid, False, q=True) + 16 * p * mid
        return {"bytes": nbytes, "flops": 2 * p * mid * mid * 17}
    if kind == "attention":
        b, rows, keys = case["batch"], case["rows"], case["prefix"] + case["suffix"]
        cells = b * 15 * rows * keys
        nbytes = b * (rows * 960 + 2 * keys * 320) * 33 / 32 + cells * (4 + 33 / 32) \
            + 4 * b * 15 * rows * 64 + 4 * rows * keys
        return {"bytes": nbytes, "flops": 2 * 2 * cells * 64}
    if kind == "gacc":
        tokens, entries = 4 * case["quads"], 4 * case["quads"] * case["slots"] * 4 * GACC_CAMERAS
        channels = 32 * case["blocks"]
        # the lists, the weights and the result; a gathered row comes from
        # the feature pool, whose rows are read many times: the pool once
        nbytes = 8 * entries + 4 * tokens * case["slots"] * case["blocks"] \
            + 4 * tokens * channels + GACC_POOL * 33 * case["blocks"]
        return {"bytes": nbytes, "flops": 2 * entries * channels * 0.9}
    return {"bytes": case["rows"] * case["cols"] * (4 + 33 / 32),
            "flops": 2 * case["rows"] * case["cols"]}


# ------------------------------------------------------------- tolerance --

def tolerance(case):
    kind = case["kind"]
    if kind in ("gacc", "encode") or case.get("mode") == "exact":
        return "exact"  # bit for bit the NPU's arithmetic
    if kind == "linear":
        # exact products, FP32 sums in another order (measured against
        # float64: up to 8e-8, FP8 inputs 5e-8; one output 4e-7); a
        # requantized byte at a rounding tie may differ
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-4}
    # a byte at a tie moves the next layer's input by one step, 1/64 of its
    # block's largest value (measured against float64: up to 2.5e-4, one
    # output 3.6e-2)
    return {"rel": 1e-3, "max": 0.1, "differ": 1e-3}


# ----------------------------------------------------------------- exact --

def _activation(x, table):
    """x T(|x|) with T from the table: index and 16-bit fraction of |x| cut
    to 21 fraction bits, 1 from 16 on; x - |x| T for negative x."""
    t = torch.from_numpy(table[512:].copy().view(np.float32).reshape(512, 2).astype(np.float64)).to(DEV)
    fixed = torch.floor(x.abs().clamp(max=16) * 2 ** 21).long()
    i = (fixed >> 16).clamp(max=511)
    v = t[i, 0] + t[i, 1] * ((fixed & 0xFFFF).double() / 65536)
    v = torch.where(x.abs() >= 16, torch.ones_like(v), v)
    return torch.where(x < 0, x - x * v, x * v)


def _through_words(y):
    q, e = _quantize(y)
    return (q * torch.exp2((e - 6).double()).unsqueeze(-1)).view(y.shape)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        m, kb, n = case["m"], case["k"] // 32, case["n"]
        out = torch.empty((case["layers"], m, n), dtype=torch.float64, device=DEV)
        for i in range(case["layers"]):
            a = _read_words(s["a"][i], m, kb, case["act"] == "fp8")
            y = a @ _read_weights(s["w"][i], n, kb).T
            if case["epilogue"] == "scale_bias":
                y = y * s["scale"][i].double() + s["bias"][i].double()
            elif case["epilogue"] == "residual":
                y = y + s["x"][i].double()
            elif case["epilogue"] == "relu_q":
                y = (y + s["bias"][i].double()).relu()
            out[i] = y
        return {"c": out, "q": None}
    if kind in ("gated_mlp", "gelu_mlp"):
        d, h = case["width"], case["hidden"]
        x, gated = s["x"].double(), kind == "gated_mlp"
        if not gated:
            x = x - x.mean(1, keepdim=True)
        y = x * torch.rsqrt(x.square().mean(1, keepdim=True) + float(np.float32(EPS))) \
            * s["gamma"].double()
        a = _through_words(y if gated else y + s["beta"].double())
        up = a @ _read_weights(s["w_up"], h, d // 32).T
        if gated:
            gate = a @ _read_weights(s["w_gate"], h, d // 32).T
            hid = _activation(gate, _table("silu")) * up
        else:
            up = _activation(up * s["s_up"].double() + s["b_up"].double(), _table("gelu"))
            hid = up
        y = _through_words(hid) @ _read_weights(s["w_down"], d, h // 32).T
        y = y + s["x"].double() if gated else y * s["s_down"].double() + s["b_down"].double()
        return {"normed": None, "up": up, "hid": None, "y": y}
    if kind == "bottleneck":
        p, mid = case["positions"], case["mid"]
        t2 = _read_words(s["cols"], p, 9 * mid // 32) @ _read_weights(s["w2"], mid, 9 * mid // 32).T
        t2 = _through_words((t2 + s["b2"].double()).relu())
        y = t2 @ _read_weights(s["w3"], 4 * mid, mid // 32).T
        y = (y + s["b3"].double() + s["residual"].double()).relu()
        return {"t1": None, "t2": None, "y": y, "y8": None}
    if kind == "attention":
        return _exact_attention(case, s)
    if kind == "gacc":
        quads, blocks, slots = case["quads"], case["blocks"], case["slots"]
        feats = s["pool"][:, :32 * blocks].contiguous().view(torch.int8).view(GACC_POOL, blocks, 32)
        scale = torch.exp2(s["pool"][:, 32 * blocks:33 * blocks].double() - 133)
        acc = torch.zeros((quads * 4, blocks, 32), dtype=torch.float64, device=DEV)
        live = (~s["out"]).double()
        for c in range(GACC_CAMERAS):
            for i in range(slots):
                w = s["w"][:, :, i // 8, :, i % 8].permute(0, 2, 1).reshape(-1, blocks).double()
                for k in range(4):
                    r = s["rows"][c, :, i, :, k].reshape(-1)
                    f = (s["bw"][c, :, i, :, k] * live[c, :, i, :, k]).reshape(-1, 1).double()
                    acc += feats[r].double() * (w * f * scale[r]).unsqueeze(-1)
        return acc.view(quads * 4, -1)
    return None


def _exact_attention(case, s):
    b, rows, keys = case["batch"], case["rows"], case["prefix"] + case["suffix"]
    pad = (rows + 3) // 4 * 4
    q = _read_words(s["q"], b * pad, 30).view(b, pad, 5, 3, 64)[:, :rows]
    k = _read_words(s["k"], b * keys, 10).view(b, keys, 5, 64)
    # V: each block of 32 tokens x 32 dimensions takes its largest scale
    # among the tokens with a nonzero value, the codes rounded to it
    w = s["v"].view(-1, 10, 144)
    code = w[:, :, :128].reshape(-1, 10, 4, 32).transpose(1, 2).reshape(b * keys // 32, 32, 10, 32)
    code = code.contiguous().view(torch.int8).double()
    e = w[:, :, 128:132].transpose(1, 2).reshape(b * keys // 32, 32, 10).double()
    any_ = (code != 0).any(-1)
    top = torch.where(any_, e, torch.full_like(e, -1)).amax(1, keepdim=True)
    top = torch.where(top < 0, torch.full_like(top, 127), top)
    shift = (top - e).unsqueeze(-1)
    v = torch.where((shift < 9) & any_.unsqueeze(-1), torch.round(code * torch.exp2(-shift)),
                    torch.zeros_like(code)) * torch.exp2(top - 133).unsqueeze(-1)
    v = v.view(b, keys, 5, 64)
    t = torch.from_numpy(_table("silu")[:512].copy().view(np.float32).reshape(512, 2)
                         .astype(np.float64)).to(DEV)
    # (plain products over float64 copies: one KV head and query at a time)
    scores = torch.zeros((b, 15, pad, keys), dtype=torch.float64, device=DEV)
    o = torch.empty((b, 15, rows, 64), dtype=torch.float64, device=DEV)
    for h in range(15):
        j, r = h // 3, h % 3
        x = q[:, :, j, r].contiguous() @ k[:, :, j].transpose(1, 2).contiguous()
        x = (x + s["mask"].double()) * 0.125
        scores[:, h, :rows] = x
        z = (x - x.amax(-1, keepdim=True)) * LOG2E
        z = torch.floor(z * 2 ** 25) / 2 ** 25
        whole = torch.floor(z)
        f = (z - whole) * 512
        i = torch.floor(f).long().clamp(0, 511)
        y = (t[i, 0] + t[i, 1] * (f - i)) * torch.exp2(whole.clamp(min=-1000))
        y = torch.where(whole < -126, torch.zeros_like(y), y)
        y = y / y.sum(-1, keepdim=True)
        o[:, h] = _through_words(y.reshape(-1, keys)).view(b, rows, keys) @ v[:, :, j].contiguous()
    return {"scores": scores, "p": None, "o": o}

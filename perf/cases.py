"""Performance cases: the calls a program makes through the public entry points, at real sizes.

One MoE layer is what this framework runs, so every case is one layer (or one of its stages)
as a serving program calls it: the views, the expert address table and the buffer structs are
made once and kept; each pass opens a segment, encodes, and commits it on the current stream.
- decode: the layer of a generation step (1 to 8 rows), sm_encode_moe_decode_layer;
- layer:  one prefill chunk, sm_encode_full_layer;
- prompt: a whole prompt through the chunk driver, sm_encode_prefill_moe_chunks;
- route:  router, top-k, grouping and gather alone, sm_encode_route_gather (a program whose
          experts run elsewhere).

Inputs: activations N(0, 1) in F16, weights N(0, 0.02) quantized to the case's block formats,
router weights N(0, 0.02) in F32, and with `zipf` > 0 a router bias that skews the experts'
load, -zipf * ln(rank) over a random order of the experts.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from __graft_entry__ import load_package

_pkg = load_package()
moe = _pkg.moe

FMT = {"Q8_0": moe.Q8_0, "Q4_K": moe.Q4_K, "Q2_K": moe.Q2_K, "F16": moe.F16, "BF16": moe.BF16}
BLOCK = {"Q8_0": (32, 34), "Q4_K": (256, 144), "Q2_K": (256, 84), "F16": (1, 2), "BF16": (1, 2)}


# Widths: (hidden, experts, top_k, expert_ff, gate_up, down, shared format). The first is the
# reference model's own; the others are this repository's benchmark and test layers.
WINDOW = dict(hidden=2560, experts=512, top_k=10, ff=640, gate_up="Q4_K", down="Q8_0", shared="F16")
FULL = dict(hidden=2048, experts=512, top_k=10, ff=512, gate_up="Q4_K", down="Q8_0", shared="F16")
LOW_BIT = dict(hidden=4096, experts=256, top_k=8, ff=1536, gate_up="Q2_K", down="Q4_K", shared="BF16")
SMALL = dict(hidden=1024, experts=64, top_k=8, ff=512, gate_up="Q2_K", down="Q4_K", shared="BF16")
Q8 = dict(hidden=2048, experts=128, top_k=10, ff=512, gate_up="Q8_0", down="Q8_0", shared="F16")
TINY = dict(hidden=256, experts=16, top_k=4, ff=256, gate_up="Q8_0", down="Q8_0", shared="F16")


def _case(kind, widths, rows, shared_ff, zipf=0.0, chunk=0, name=None):
    c = dict(kind=kind, rows=rows, shared_ff=shared_ff, zipf=zipf, chunk=chunk, **widths)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # One generated token: the latency of a single user's decode step.
        _case("decode", WINDOW, 1, 640, name="decode_1"),
        # A full decode window (speculative rows, or eight users batched).
        _case("decode", WINDOW, 8, 640, name="decode_8"),
        # A part-filled window on the low-bit layer with its BF16 shared expert.
        _case("decode", LOW_BIT, 4, 1536, name="decode_low_bit_4"),
        # The smallest prefill call: launches and host time.
        _case("layer", TINY, 64, 0, name="prefill_tiny_64"),
        # A short chat turn: few rows for each of many experts.
        _case("layer", FULL, 100, 512, name="prefill_turn_100"),
        # A short prompt on a model of few experts, low-bit weights.
        _case("layer", SMALL, 333, 512, name="prefill_small_333"),
        # Eight-bit experts, a ragged chunk (the tail of a prompt).
        _case("layer", Q8, 513, 512, name="prefill_q8_513"),
        # A ragged chunk at the reference model's own expert widths.
        _case("layer", WINDOW, 1000, 0, name="prefill_window_1000"),
        # The benchmark layer: one 2048-token chunk.
        _case("layer", FULL, 2048, 512, name="prefill_2048"),
        # A large chunk with skewed experts: hot experts take thousands of rows, others few.
        _case("layer", FULL, 8192, 512, zipf=1.1, name="prefill_skew_8192"),
        # A long prompt through the chunk driver, low-bit weights.
        _case("prompt", LOW_BIT, 16384, 1536, chunk=4096, name="prompt_16384"),
        # Routing and dispatch alone.
        _case("route", FULL, 4096, 0, name="route_4096"),
    ]


def _log_rows(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "layer", "layer", "layer", "layer", "prompt", "route"])
    if kind == "decode":
        w, sf = rng.choice([(WINDOW, 640), (FULL, 512), (LOW_BIT, 1536), (SMALL, 512)])
        return _case(kind, w, rng.randint(1, 8), sf, zipf=rng.choice([0.0, 1.1]))
    if kind == "layer":
        w, sf, hi = rng.choice([(FULL, 512, 8192), (WINDOW, 0, 4096), (LOW_BIT, 1536, 4096), (SMALL, 512, 4096),
                                (Q8, 512, 4096), (TINY, 0, 1024)])
        return _case(kind, w, _log_rows(rng, 9, hi), sf, zipf=rng.choice([0.0, 0.6, 1.1]))
    if kind == "prompt":
        w, sf = rng.choice([(FULL, 512), (WINDOW, 0), (LOW_BIT, 1536)])
        return _case(kind, w, _log_rows(rng, 1024, 8192), sf, zipf=rng.choice([0.0, 0.6]),
                     chunk=rng.choice([512, 1024, 2048, 4096]))
    w = rng.choice([FULL, WINDOW, LOW_BIT, SMALL])
    return _case(kind, w, _log_rows(rng, 9, 8192), 0, zipf=rng.choice([0.0, 1.1]))


# ---- inputs ---------------------------------------------------------------------------------

def _quantize(fmt, x):
    """x F32 [n, block values] -> bytes [n, block bytes] (ggml block layouts)."""
    n = x.shape[0]
    if fmt == "Q8_0":
        d = (x.abs().amax(1, keepdim=True) / 127.0)
        q = torch.round(x / d).clamp_(-127, 127).to(torch.int8)
        return torch.cat([d.half().view(torch.uint8), q.view(torch.uint8)], 1)
    sub, top, code = (8, 63, 15) if fmt == "Q4_K" else (16, 15, 3)
    xs = x.view(n, sub, -1)
    lo, hi = xs.amin(2).clamp_(max=0.0), xs.amax(2)
    sc, mn = (hi - lo) / code, -lo
    d = (sc.amax(1, keepdim=True) / top).half()
    dmin = (mn.amax(1, keepdim=True) / top).half()
    ls = torch.round(sc / d.float()).clamp_(0, top)
    lm = torch.round(mn / dmin.float()).clamp_(0, top)
    dl, ml = d.float() * ls, dmin.float() * lm
    q = torch.round((xs + ml[:, :, None]) / dl[:, :, None]).clamp_(0, code).to(torch.uint8)
    ls, lm = ls.to(torch.uint8), lm.to(torch.uint8)
    head = torch.cat([d.view(torch.uint8), dmin.view(torch.uint8)], 1)
    if fmt == "Q4_K":
        scales = torch.cat([ls[:, :4] | ((ls[:, 4:] >> 4) << 6), lm[:, :4] | ((lm[:, 4:] >> 4) << 6),
                            (ls[:, 4:] & 15) | ((lm[:, 4:] & 15) << 4)], 1)
        q = q.view(n, 4, 2, 32)  # 64-value groups: low nibbles, then high nibbles
        return torch.cat([head, scales, (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(n, 128)], 1)
    q = q.view(n, 2, 4, 32)  # 128-value halves of four 2-bit planes
    qs = q[:, :, 0] | (q[:, :, 1] << 2) | (q[:, :, 2] << 4) | (q[:, :, 3] << 6)
    return torch.cat([ls | (lm << 4), qs.reshape(n, 64), head], 1)


def _dequantize(fmt, b, values):
    """Bytes [rows, row bytes] -> F64 [rows, values], d * code (- min) exactly."""
    rows = b.shape[0]
    if fmt in ("F16", "BF16"):
        return b.view(torch.float16 if fmt == "F16" else torch.bfloat16).double()
    bv, bb = BLOCK[fmt]
    blk = b.view(rows * (values // bv), bb)
    f16 = lambda s: s.contiguous().view(torch.float16).double()  # noqa: E731
    if fmt == "Q8_0":
        return (f16(blk[:, :2]) * blk[:, 2:].contiguous().view(torch.int8).double()).view(rows, values)
    if fmt == "Q4_K":
        d, dmin, s = f16(blk[:, 0:2]), f16(blk[:, 2:4]), blk[:, 4:16]
        ls = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        lm = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = blk[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
    else:
        d, dmin = f16(blk[:, 80:82]), f16(blk[:, 82:84])
        ls, lm = blk[:, :16] & 15, blk[:, :16] >> 4
        qs = blk[:, 16:80].view(-1, 2, 1, 32)
        q = torch.cat([(qs >> (2 * j)) & 3 for j in range(4)], 2).view(-1, 16, 16)
    w = q.double() * (d * ls.double())[:, :, None] - (dmin * lm.double())[:, :, None]
    return w.view(rows, values)


def _weights(fmt, gen, matrices, rows, values):
    """Quantized N(0, 0.02) weights: bytes [matrices, rows * row bytes]."""
    bv, bb = BLOCK[fmt]
    per = rows * (values // bv)
    out = torch.empty(matrices, per * bb, dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 26) // (rows * values))
    for m in range(0, matrices, step):
        n = min(step, matrices - m)
        x = torch.randn(n * per, bv, generator=gen, device="cuda") * 0.02
        out[m:m + n] = _quantize(fmt, x).view(n, per * bb)
    return out


def _inputs(case, seed):
    """The tensors a program holds before the call, made on the GPU from the seed alone."""
    gen = torch.Generator("cuda").manual_seed(seed)
    T, d, E, I, Is = case["rows"], case["hidden"], case["experts"], case["ff"], case["shared_ff"]
    t = dict(x=torch.randn(T, d, generator=gen, device="cuda").half(),
             router=torch.randn(E, d, generator=gen, device="cuda") * 0.02, bias=None)
    if case["zipf"] > 0:
        rank = torch.randperm(E, generator=gen, device="cuda").double() + 1.0
        t["bias"] = (-case["zipf"] * torch.log(rank)).float()
    if case["kind"] != "route":
        t["gate"] = _weights(case["gate_up"], gen, E, I, d)
        t["up"] = _weights(case["gate_up"], gen, E, I, d)
        t["down"] = _weights(case["down"], gen, E, d, I)
        if Is:
            dt = torch.float16 if case["shared"] == "F16" else torch.bfloat16
            for name, shape in (("sh_gate", (Is, d)), ("sh_up", (Is, d)), ("sh_down", (d, Is)), ("sh_vec", (d,))):
                t[name] = (torch.randn(*shape, generator=gen, device="cuda") * 0.02).to(dt)
    return t


# ---- what a program keeps: context, views, buffers ---------------------------------------------

class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, s.t = case, _inputs(case, seed)
    s.ctx = moe.Context(torch.cuda.current_device())
    s.bufs = {}
    T, d, E, K, I, Is = (case[k] for k in ("rows", "hidden", "experts", "top_k", "ff", "shared_ff"))
    C = min(case["chunk"], T) if case["kind"] == "prompt" else T  # rows of one layer call
    N = C * K
    s.shape = moe.Shape(C, d, E, K, I, Is)

    def view(name, tensor=None, length=None):
        if tensor is not None:
            s.bufs[name] = (tensor, s.ctx.register_ptr(tensor.data_ptr(), tensor.numel() * tensor.element_size()))
        return s.bufs[name][1].view() if length is None else s.bufs[name][1].view(*length)

    def buf(name, *shape, dtype=torch.float32, zero=False):
        return view(name, (torch.zeros if zero else torch.empty)(*shape, dtype=dtype, device="cuda"))

    null = moe.NULL_VIEW
    s.formats = moe.LayerFormats(FMT[case["gate_up"]], FMT[case["down"]], FMT[case["shared"]])
    x = view("x", s.t["x"])
    router = view("router", s.t["router"])
    bias = view("bias", s.t["bias"]) if s.t["bias"] is not None else null
    logits, ids, weights = buf("logits", C, E), buf("ids", C, K, dtype=torch.int32), buf("weights", C, K)
    if case["kind"] != "route":
        gate, up, down = (view(n, s.t[n]) for n in ("gate", "up", "down"))
        table = []
        for e in range(E):
            table += [s.t[n].data_ptr() + e * s.t[n].shape[1] for n in ("gate", "up", "down")]
        s.gu = moe.ExpertTable(table, buf("snap_gu", E * 3, dtype=torch.int64), [gate, up])
        s.dn = moe.ExpertTable(table, buf("snap_dn", E * 3, dtype=torch.int64), [down])
    shared = moe.SharedBuffers()
    if Is and case["kind"] != "route":
        hdt = torch.float32 if case["kind"] == "decode" else torch.float16
        shared = moe.SharedBuffers(x, view("sh_gate", s.t["sh_gate"]), view("sh_up", s.t["sh_up"]),
                                   view("sh_down", s.t["sh_down"]), view("sh_vec", s.t["sh_vec"]),
                                   buf("sh_hidden", C, Is, dtype=hdt), buf("sh_out", C, d), buf("sh_logit", C))
    out = buf("out", T, d) if case["kind"] != "route" else null
    if case["kind"] == "decode":
        plans = buf("plans", moe.MOE_PLAN_BYTES, dtype=torch.uint8)
        xq = buf("xq", moe.q8_1_bytes(C, d), dtype=torch.uint8)
        routed = moe.MoeRoutedFFNBuffers(s.gu.struct, s.dn.struct, xq, plans, buf("gate_rows", N, I),
                                         buf("up_rows", N, I), buf("hidden", N, I),
                                         buf("hq", moe.q8_1_bytes(N, I), dtype=torch.uint8), buf("parts", N, d),
                                         buf("status", 4, dtype=torch.int32, zero=True))
        s.b = moe.DecodeLayerBuffers(x, router, bias, logits, ids, weights, null, null, plans, 0, xq, routed, shared, out)
        return s
    hist = buf("hist", moe.histogram_bytes(s.shape) // 4, dtype=torch.int32)
    plan = buf("plan", moe.PLAN_SLOT_BYTES // 4, dtype=torch.int32)
    tiles = buf("tiles", moe.tiles_bytes(s.shape) // 4, dtype=torch.int32)
    src, dst = buf("src", N, dtype=torch.int32), buf("dst", N, dtype=torch.int32)
    xs = buf("xs", N, d, dtype=torch.float16)
    cx = x if case["kind"] != "prompt" else view("chunk_x", torch.empty(C, d, dtype=torch.float16, device="cuda"))
    s.rg = moe.RouteGatherBuffers(cx, router, logits, ids, weights, hist, plan, tiles, src, dst, xs, bias)
    if case["kind"] == "route":
        return s
    if Is:
        shared.mixed_h = cx
    chunk_out = out if case["kind"] == "layer" else buf("chunk_out", C, d)
    buf("status", 8, dtype=torch.int32, zero=True)
    hidden, parts = buf("hidden", N, I, dtype=torch.float16), buf("parts", N, d)
    s.b = moe.LayerBuffers(
        s.rg, shared,
        moe.GateUpBuffers(s.gu.struct, xs, plan, tiles, hidden, view("status", length=(0, 4))),
        moe.DownBuffers(s.dn.struct, hidden, plan, tiles, dst, parts, view("status", length=(4, 4))),
        moe.CombineBuffers(parts, weights, shared.output if Is else null, shared.gate_logit if Is else null, chunk_out))
    if case["kind"] == "prompt":
        s.schedule, err = moe.build_chunk_schedule(0, T, C)
        assert s.schedule is not None, err
        s.x_view, s.out_view = x, out
    return s


def run(s):
    kind = s.case["kind"]
    seg = s.ctx.segment()
    if kind == "decode":
        ok, err = seg.encode_moe_decode_layer(s.shape, s.formats, s.b)
    elif kind == "layer":
        ok, err = seg.encode_prefill_moe_full_mode_layer(s.shape, s.formats, s.b)
    elif kind == "prompt":
        ok, err = seg.encode_prefill_moe_chunks(s.schedule, s.shape, s.formats, s.x_view, s.out_view, s.b)
    else:
        ok, err = seg.encode_prefill_moe_full_mode_route_gather(s.shape, s.rg)
    if not ok:
        seg.abort()
        raise RuntimeError(err)
    seg.commit(torch.cuda.current_stream().cuda_stream)
    names = {"decode": ("out", "logits", "ids", "weights"), "layer": ("out", "logits", "ids", "weights"),
             "prompt": ("out",), "route": ("logits", "ids", "weights", "src", "dst", "xs")}[kind]
    return {n: s.bufs[n][0] for n in names}


# ---- work, tolerances, exact results ------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _used_experts(rows, experts, top_k, hidden, zipf):
    """Experts that `rows` tokens select (a fixed simulation of the router's logits)."""
    rng = np.random.default_rng(1)
    bias = -zipf * np.log(np.arange(1, experts + 1))
    used = np.zeros(experts, bool)
    for r in range(0, min(rows, 8192), 1024):
        z = rng.standard_normal((min(1024, rows - r), experts)) * (0.02 * math.sqrt(hidden)) + bias
        used[np.argpartition(-z, top_k - 1, axis=1)[:, :top_k] if top_k < experts else slice(None)] = True
    return int(used.sum())


def work(case):
    T, d, E, K, I, Is = (case[k] for k in ("rows", "hidden", "experts", "top_k", "ff", "shared_ff"))
    N = T * K
    byts = T * d * 2 + E * d * 4 + T * E * 4 + N * 8
    flops = 2.0 * T * E * d
    if case["kind"] == "route":
        return {"bytes": byts + N * 8 + N * d * 2, "flops": flops}
    row = lambda fmt, n: n // BLOCK[fmt][0] * BLOCK[fmt][1]  # noqa: E731
    if case["kind"] == "prompt":
        byts -= T * E * 4 + N * 8
    byts += T * d * 4
    byts += _used_experts(T, E, K, d, case["zipf"]) * (2 * I * row(case["gate_up"], d) + d * row(case["down"], I))
    flops += 6.0 * N * I * d
    if Is:
        byts += 3 * Is * d * 2 + d * 2
        flops += 6.0 * T * Is * d + 2.0 * T * d
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    # Four times what the path showed against `exact` (2-norm): 2e-5 in prefill (F16 hidden rows
    # that round the other way after an F32 sum in another order), 7e-4 in decode (Q8_1 codes of
    # the hidden rows likewise), 2e-3 over a whole prompt's 16384 tokens, where a token or two
    # has an expert in the tenth place that F32 logits cannot tell from the eleventh.
    # ids: two experts whose logits differ by less than the F32 rounding may swap.
    return {"rel": {"decode": 3e-3, "prompt": 8e-3}.get(case["kind"], 1e-4), "differ": 1e-3}


def _q8_1(v):
    """Q8_1 blocks of 32 as the decode path stores activations: F16 scale amax / 127, codes
    rounded half away from zero."""
    b = v.view(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127.0
    q = torch.where(d > 0, b / d, torch.zeros_like(b))
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return (q * d.half().double()).view(v.shape)


def exact(case, seed):
    """The layer in 64 bits: plain products on the dequantized weights. Values that the layer
    stores in 16 or 8 bits by definition (F16 weights and hidden rows in prefill, Q8_1
    activations in decode) are rounded where they are stored; every sum is in F64."""
    t = _inputs(case, seed)
    T, d, E, K, I, Is = (case[k] for k in ("rows", "hidden", "experts", "top_k", "ff", "shared_ff"))
    decode = case["kind"] == "decode"
    x = t["x"].double()
    logits = x @ t["router"].double().t()
    if t["bias"] is not None:
        logits += t["bias"].double()
    p = torch.softmax(logits, 1)
    # the larger probability first, the lower expert on ties
    w, ids = torch.sort(p, dim=1, descending=True, stable=True)
    w, ids = w[:, :K].contiguous(), ids[:, :K].contiguous()
    w = w / w.sum(1, keepdim=True).clamp_(min=2.0 ** -14)
    if case["kind"] == "route":
        # an id swap moves every later row, so the dispatch itself has no 64-bit counterpart
        return {"logits": logits, "ids": ids, "weights": w, "src": None, "dst": None, "xs": None}
    w16 = (lambda m: m) if decode else (lambda m: m.half().double())
    h16 = _q8_1 if decode else (lambda m: m.half().double())
    xe = _q8_1(x) if decode else x
    out = torch.zeros(T, d, dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        tok, rank = torch.nonzero(ids == e, as_tuple=True)
        wg = w16(_dequantize(case["gate_up"], t["gate"][e].view(I, -1), d))
        wu = w16(_dequantize(case["gate_up"], t["up"][e].view(I, -1), d))
        wd = w16(_dequantize(case["down"], t["down"][e].view(d, -1), I))
        rows = xe[tok]
        h = h16(torch.nn.functional.silu(rows @ wg.t()) * (rows @ wu.t()))
        out.index_add_(0, tok, (h @ wd.t()) * w[tok, rank][:, None])
    if Is:
        sg, su, sd, sv = (w16(t[n].double()) for n in ("sh_gate", "sh_up", "sh_down", "sh_vec"))
        h = torch.nn.functional.silu(x @ sg.t()) * (x @ su.t())
        h = h if decode else h.half().double()
        out += (h @ sd.t()) * torch.sigmoid(x @ sv)[:, None]
    if case["kind"] == "prompt":
        return {"out": out}
    return {"out": out, "logits": logits, "ids": ids, "weights": w}

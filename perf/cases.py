"""The work that a program has this library do, as timed cases.

A 64-layer hybrid transformer (hidden 5120, feed-forward 17408, QKV 12288,
attention output 6144 -> 5120, vocabulary 248320) is served one token at a time
(decode), a few sequences at a time (batched decode) and in chunks of up to
1024 prompt tokens (prefill). Its weights are Q4_K / Q6_K against Q8
activations, the same Q4_K bytes against BF16 activations, FP8 (E4M3) mixer
projections, NVFP4 gate/up projections and a Q8G32 vocabulary head. Every case
is one layer step through the entry points that such a program calls, with
freshly seeded weights that follow their format's usual fit and activations
with a few large channels.

``listed()`` names the cases, ``draw()`` makes more of the same ranges,
``prepare()`` makes what the program holds before the call, ``run()`` is one
pass, ``exact()`` the same result in 64 bits from plain torch, ``work()`` the
bytes and operations that cannot be avoided and ``tolerance()`` how far two
correct implementations may differ.
"""
from __future__ import annotations

import math

import torch

from qw38_amd import ops
from qw38_amd._lib import LAYOUT_Q4K_SEQ

HIDDEN, FFN, QKV, ATTN, VOCAB = 5120, 17408, 12288, 6144, 248320
EPS = 1e-6
ROWS = 4096  # weight rows made or contracted at a time


def listed():
    return [
        # One token through the attention output projection, Q8 pack included: the smallest call.
        dict(name="q8_out_decode_1", kind="q8_project", quant="q4_k", n=HIDDEN, k=ATTN, m=1, residual=True),
        # Six sequences decoding together through the QKV projection.
        dict(name="q8_qkv_decode_6", kind="q8_project", quant="q4_k", n=QKV, k=HIDDEN, m=6, residual=False),
        # A whole prompt chunk through the QKV projection.
        dict(name="q8_qkv_prefill_512", kind="q8_project", quant="q4_k", n=QKV, k=HIDDEN, m=512, residual=False),
        # The feed-forward block of one decoded token (Q4_K gate/up, Q6_K down).
        dict(name="q8_mlp_decode_1", kind="q8_mlp", m=1),
        # The feed-forward block of a prompt's ragged last chunk.
        dict(name="q8_mlp_prefill_387", kind="q8_mlp", m=387),
        # Gate and up of one decoded token on BF16 activations, the route without Q8.
        dict(name="bf16_gate_up_decode", kind="decode", layout="q4_k", n=FFN, k=HIDDEN, epilogue="swiglu"),
        # The BF16 feed-forward block of a ragged prompt chunk.
        dict(name="bf16_mlp_prefill_300", kind="prefill_mlp", layout="q4_k", m=300),
        # The FP8 QKV projection of one decoded token.
        dict(name="fp8_qkv_decode", kind="decode", layout="fp8", n=QKV, k=HIDDEN, epilogue="bf16"),
        # The FP8 QKV projection of a prompt chunk, activation pack included.
        dict(name="fp8_qkv_prefill_512", kind="fp8_project", n=QKV, k=HIDDEN, m=512, epilogue="bf16"),
        # NVFP4 gate and up of one decoded token.
        dict(name="nvfp4_gate_up_decode", kind="decode", layout="nvfp4", n=FFN, k=HIDDEN, epilogue="swiglu"),
        # The feed-forward block with NVFP4 gate/up on the largest prompt chunk.
        dict(name="nvfp4_mlp_prefill_1024", kind="prefill_mlp", layout="nvfp4", m=1024),
        # The vocabulary head of one decoded token: the most bytes of a single call.
        dict(name="head_decode", kind="decode", layout="q8g32", n=VOCAB, k=HIDDEN, epilogue="fp32"),
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer in [lo, hi], a multiple of step, spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi // step * step, int(v) // step * step))


def draw(rng):
    kind = rng.choice(["q8_project", "q8_project", "q8_mlp", "decode", "decode", "prefill_mlp", "fp8_project"])
    if kind == "q8_project":
        k = _log_int(rng, 1024, FFN, 256)
        n = min(_log_int(rng, 1024, 34816), 34816 * HIDDEN // k)
        m = min(_log_int(rng, 1, 2048), 10**11 // (n * k))
        return dict(kind=kind, quant=rng.choice(["q4_k", "q4_k", "q6_k"]), n=n, k=k, m=m,
                    residual=rng.random() < 0.5)
    if kind == "q8_mlp":
        return dict(kind=kind, m=_log_int(rng, 1, 512))
    if kind == "prefill_mlp":
        return dict(kind=kind, layout=rng.choice(["q4_k", "nvfp4"]), m=_log_int(rng, 2, 1024))
    if kind == "fp8_project":
        return dict(kind=kind, n=_log_int(rng, 1024, QKV, 128), k=_log_int(rng, 1024, ATTN, 256),
                    m=_log_int(rng, 2, 1024), epilogue=rng.choice(["bf16", "fp32", "residual"]))
    layout = rng.choice(["q4_k", "fp8", "nvfp4", "q8g32"])
    epilogue = rng.choice(["bf16", "fp32", "residual"] + ([] if layout == "fp8" else ["swiglu"]))
    if layout == "q8g32":
        return dict(kind=kind, layout=layout, n=_log_int(rng, 4096, VOCAB if epilogue != "swiglu" else VOCAB // 2),
                    k=_log_int(rng, 1024, HIDDEN, 32), epilogue=epilogue)
    # a matrix of rows that one projection or a gate/up pair of the model has
    return dict(kind=kind, layout=layout, n=_log_int(rng, 1024, FFN, {"q4_k": 1, "fp8": 128, "nvfp4": 8}[layout]),
                k=_log_int(rng, 1024, ATTN, 256), epilogue=epilogue)


# ---- weights: rows of a normal matrix fitted to each format ------------------
# Each maker yields (first row, the format's device bytes, the float64 operand
# rows or None): the operands are only built for exact().

def _rows(gen, n, k):
    for r in range(0, n, ROWS):
        yield r, torch.randn(min(ROWS, n - r), k, generator=gen, device="cuda") / math.sqrt(k)


def _q4_k(gen, n, k, operands):
    """GGML Q4_K super-blocks: 6-bit scales and minima of eight 32-groups."""
    for r, w in _rows(gen, n, k):
        rows = w.shape[0]
        w = w.view(rows, k // 256, 8, 32)
        lo = w.amin(-1).clamp(max=0)
        scale, low = (w.amax(-1) - lo) / 15, -lo
        d = (scale.amax(-1, keepdim=True) / 63).half()
        dmin = (low.amax(-1, keepdim=True) / 63).half()
        s = (scale / d.float()).round().clamp(0, 63)
        m = (low / dmin.float()).round().clamp(0, 63)
        ds, dm = d.float() * s, dmin.float() * m
        q = ((w + dm[..., None]) / ds[..., None].clamp(min=1e-30)).round().clamp(0, 15).to(torch.uint8)
        if operands:
            yield r, None, (ds.double(), dm.double(), q.double())
            continue
        si, mi = s.to(torch.int32), m.to(torch.int32)
        head = torch.cat([si[..., :4] | (si[..., 4:] >> 4 << 6), mi[..., :4] | (mi[..., 4:] >> 4 << 6),
                          (si[..., 4:] & 15) | ((mi[..., 4:] & 15) << 4)], -1).to(torch.uint8)
        qs = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(rows, k // 256, 128)
        yield r, torch.cat([d.view(torch.uint8), dmin.view(torch.uint8), head, qs], -1).view(-1), None


def _q6_k(gen, n, k, operands):
    """GGML Q6_K super-blocks: int8 scales of sixteen 16-groups."""
    for r, w in _rows(gen, n, k):
        rows = w.shape[0]
        w = w.view(rows, k // 256, 16, 16)
        top = w.abs().amax(-1) / 31
        d = (top.amax(-1, keepdim=True) / 127).half()
        s = (top / d.float()).round().clamp(1, 127)
        ds = d.float() * s
        q = (w / ds[..., None]).round().clamp(-32, 31)
        if operands:
            yield r, None, (ds.double(), q.double())
            continue
        c = (q + 32).to(torch.uint8).view(rows, k // 256, 2, 4, 32)  # [half][part][l]
        ql = torch.cat([(c[..., 0, :] & 15) | (c[..., 2, :] << 4), (c[..., 1, :] & 15) | (c[..., 3, :] << 4)], -1)
        h = c >> 4
        qh = h[..., 0, :] | (h[..., 1, :] << 2) | (h[..., 2, :] << 4) | (h[..., 3, :] << 6)
        yield r, torch.cat([ql.flatten(2), qh.flatten(2), s.to(torch.int8).view(torch.uint8),
                            d.view(torch.uint8)], -1).view(-1), None


def _fp8(gen, n, k, operands):
    """E4M3 codes with one FP32 scale per 128 x 128 block."""
    for r, w in _rows(gen, n, k):
        rows = w.shape[0]
        b = w.view(rows // 128, 128, k // 128, 128)
        s = b.abs().amax((1, 3), keepdim=True) / 448
        c = (b / s).to(torch.float8_e4m3fn)
        s = s[:, 0, :, 0]
        if operands:
            yield r, None, (c.double() * s.double()[:, None, :, None]).view(rows, k)
        else:
            yield r, (c.view(rows, k).view(torch.uint8), s.t()), None


E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _e2m1(v):
    """Codes of the nearest E2M1 magnitudes, ties to the even code, sign in bit 3."""
    a = v.abs()
    c = (a > 0.25).to(torch.uint8)
    for edge, up in ((0.75, True), (1.25, False), (1.75, True), (2.5, False), (3.5, True), (5.0, False)):
        c += (a >= edge) if up else (a > edge)
    return c | ((v < 0).to(torch.uint8) << 3)


def _e2m1_values(c):
    table = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=c.device)
    return table[c.long()]


def _nvfp4_blocks(v):
    """(E4M3 scale codes, E2M1 codes) of [rows][blocks][16] values."""
    peak = v.abs().amax(-1)
    s = (peak / 6).to(torch.float8_e4m3fn).view(torch.uint8)
    s = torch.where((s == 0) & (peak != 0), torch.ones_like(s), s)
    return s, _e2m1(v / s.view(torch.float8_e4m3fn).float()[..., None].clamp(min=2.0**-20))


NVFP4_FACTOR = 2.0**-14  # block peaks / 6 of these weights then fall into E4M3's range


def _nvfp4(gen, n, k, operands):
    for r, w in _rows(gen, n, k):
        s, c = _nvfp4_blocks((w / NVFP4_FACTOR).view(-1, k // 16, 16))
        if operands:
            f = s.view(torch.float8_e4m3fn).double() * NVFP4_FACTOR
            yield r, None, (f[..., None] * _e2m1_values(c)).view(-1, k)
        else:
            c = c.view(-1, k)
            yield r, (c[:, 0::2] | (c[:, 1::2] << 4), s), None


def _q8g32(gen, n, k, operands):
    """int8 codes and FP16 scales of 32-groups."""
    for r, w in _rows(gen, n, k):
        w = w.view(w.shape[0], k // 32, 32)
        s = (w.abs().amax(-1) / 127).half()
        c = (w / s.float()[..., None]).round().clamp(-127, 127)
        if operands:
            yield r, None, (c * s.float()[..., None]).bfloat16().double().view(-1, k)
        else:
            yield r, (c.to(torch.int8).view(-1, k), s), None


MAKERS = {"q4_k": _q4_k, "q6_k": _q6_k, "fp8": _fp8, "nvfp4": _nvfp4, "q8g32": _q8g32}


def _generator(seed, salt):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 64 + salt)
    return gen


def _weight(layout, n, k, seed, salt):
    """The device-resident weight that a loader leaves behind."""
    parts = MAKERS[layout](_generator(seed, salt), n, k, False)
    if layout in ("q4_k", "q6_k"):
        blocks = torch.empty(n * (k // 256) * (144 if layout == "q4_k" else 210), dtype=torch.uint8, device="cuda")
        at = 0
        for _, b, _ in parts:
            blocks[at:at + b.numel()] = b
            at += b.numel()
        return (ops.upload_q4k_blocks(blocks, n, k, layout=LAYOUT_Q4K_SEQ) if layout == "q4_k"
                else ops.upload_q6k_blocks(blocks, n, k))
    if layout == "fp8":
        codes = torch.empty(n, k, dtype=torch.uint8, device="cuda")
        scales = torch.empty(k // 128, n // 128, device="cuda")
        for r, (c, s), _ in parts:
            codes[r:r + c.shape[0]] = c
            scales[:, r // 128:r // 128 + s.shape[1]] = s
        return codes, scales
    if layout == "nvfp4":
        pn = (n + 127) // 128 * 128
        codes = torch.empty(n, k // 2, dtype=torch.uint8, device="cuda")
        s = torch.zeros(pn, k // 16, dtype=torch.uint8, device="cuda")
        for r, (c, sc), _ in parts:
            codes[r:r + c.shape[0]] = c
            s[r:r + c.shape[0]] = sc
        # 128-row stripes of 512-byte chunks ordered (row % 32, row / 32, block % 4)
        s = s.view(pn // 128, 4, 32, k // 64, 4).permute(0, 3, 2, 1, 4).reshape(-1)
        head = torch.zeros(64, device="cuda")
        head[0] = NVFP4_FACTOR
        return ops.nvfp4_weight(codes, torch.cat([head.view(torch.uint8), s]), n, k)
    pn, pk = ops.pad_n(n), ops.pad_k(k)  # q8g32: 8-row x K256 tiles
    codes = torch.zeros(pn // 8, pk // 256, 8, 256, dtype=torch.int8, device="cuda")
    scales = torch.zeros(pn // 8, pk // 256, 8, 8, dtype=torch.float16, device="cuda")
    pad = torch.nn.functional.pad
    for r, (c, s), _ in parts:
        rows = (c.shape[0] + 7) // 8 * 8
        c = pad(c, (0, pk - k, 0, rows - c.shape[0])).view(rows // 8, 8, pk // 256, 256)
        s = pad(s, (0, (pk - k) // 32, 0, rows - s.shape[0])).view(rows // 8, 8, pk // 256, 8)
        codes[r // 8:(r + rows) // 8] = c.transpose(1, 2)
        scales[r // 8:(r + rows) // 8] = s.transpose(1, 2)
    return ops.dense_weight(ops.DECODE_LAYOUT_Q8G32, codes.view(-1).view(torch.uint8),
                            scales.view(-1).view(torch.uint8), n, k)


# ---- activations -------------------------------------------------------------

def _tokens(seed, m, k):
    """Rows of a normalized hidden state: one channel in a hundred is 20 times larger."""
    gen = _generator(seed, 0)
    x = torch.randn(m, k, generator=gen, device="cuda")
    x[:, torch.randperm(k, generator=gen, device="cuda")[:max(1, k // 100)]] *= 20
    return x


def _gamma(seed):
    return (torch.randn(HIDDEN, generator=_generator(seed, 7), device="cuda") * 0.1).bfloat16()


def _residual(seed, m, n):
    return torch.randn(m, n, generator=_generator(seed, 8), device="cuda")


EPILOGUE = {"bf16": ops.DECODE_STORE_BF16, "fp32": ops.DECODE_STORE_FP32,
            "residual": ops.DECODE_RESIDUAL_ADD_FP32, "swiglu": ops.DECODE_SWIGLU_BF16}


def _output(case, m):
    kind = torch.bfloat16 if case["epilogue"] in ("bf16", "swiglu") else torch.float32
    return torch.empty(m, case["n"], dtype=kind, device="cuda")


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "q8_project":
        m, n, k = case["m"], case["n"], case["k"]
        s["weight"] = _weight(case["quant"], n, k, seed, 1)
        s["x"] = _tokens(seed, m, k).bfloat16()
        s["q8"] = ops.Q8Input.empty(m, k)
        s["failure"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["residual"] = _residual(seed, m, n) if case["residual"] else None
        s["out"] = torch.empty(m, n, device="cuda")
    elif kind == "q8_mlp":
        m = case["m"]
        s["weights"] = (_weight("q4_k", FFN, HIDDEN, seed, 1), _weight("q4_k", FFN, HIDDEN, seed, 2),
                        _weight("q6_k", HIDDEN, FFN, seed, 3))
        s["h"], s["gamma"] = _tokens(seed, m, HIDDEN), _gamma(seed)
        s["workspace"] = torch.empty(ops.q8_mlp_workspace_bytes(m), dtype=torch.uint8, device="cuda")
        s["failure"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["out"] = torch.empty(m, HIDDEN, device="cuda")
    elif kind == "prefill_mlp":
        m = case["m"]
        s["weights"] = (_weight(case["layout"], FFN, HIDDEN, seed, 1), _weight(case["layout"], FFN, HIDDEN, seed, 2),
                        _weight("q4_k", HIDDEN, FFN, seed, 3))
        s["h"], s["gamma"] = _tokens(seed, m, HIDDEN), _gamma(seed)
        s["workspace"] = torch.empty(ops.prefill_mlp_workspace_bytes(m), dtype=torch.uint8, device="cuda")
        s["out"] = torch.empty(m, HIDDEN, device="cuda")
    elif kind == "fp8_project":
        m, n, k = case["m"], case["n"], case["k"]
        pm = (m + 127) // 128 * 128
        s["weight"] = ops.fp8_weight_struct(*_weight("fp8", n, k, seed, 1), n, k)
        s["x"] = _tokens(seed, m, k).bfloat16()
        s["codes"] = torch.empty(pm, k, dtype=torch.uint8, device="cuda")
        s["scales"] = torch.empty(k // 128, pm, device="cuda")
        s["input"] = ops.fp8_input_struct(s["codes"], s["scales"], pm, k)
        s["residual"] = _residual(seed, m, n) if case["epilogue"] == "residual" else None
        s["out"] = _output(case, m)
    else:  # decode: one token through decode_mmv's descriptors
        n, k, layout, epi = case["n"], case["k"], case["layout"], EPILOGUE[case["epilogue"]]
        x = _tokens(seed, 1, k).bfloat16()
        s["out"] = _output(case, 1)
        residual = _residual(seed, 1, n) if case["epilogue"] == "residual" else None

        def desc(salt, out):
            w = _weight(layout, n, k, seed, salt)
            if layout == "fp8":
                return ops.fp8_decode_desc(*w, n, k, x, out, epi, residual)
            return (ops.nvfp4_decode_desc if layout == "nvfp4" else ops.decode_desc)(w, x, out, epi, residual)
        s["a"] = desc(1, s["out"])
        s["b"] = desc(2, None) if case["epilogue"] == "swiglu" else None
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "q8_project":
        ops.pack_q8(s["x"], s["q8"], s["failure"])
        ops.q4k_q8_project(s["weight"], s["q8"], s["out"], residual=s["residual"])
    elif kind == "q8_mlp":
        ops.q4k_q8_mlp(*s["weights"], s["h"], s["gamma"], EPS, s["out"], case["m"], s["workspace"],
                       pending_failure=s["failure"])
    elif kind == "prefill_mlp":
        ops.prefill_mlp(*s["weights"], s["h"], s["gamma"], EPS, s["out"], case["m"], s["workspace"])
    elif kind == "fp8_project":
        ops.pack_fp8(s["x"], case["m"], case["k"], s["codes"], s["scales"])
        ops.fp8_project(s["weight"], s["input"], case["m"], s["out"], EPILOGUE[case["epilogue"]], s["residual"])
    elif s["b"] is not None:
        ops.decode_mmv_paired(s["a"], s["b"])
    else:
        ops.decode_mmv(s["a"])
    return s["out"]


# ---- bytes and operations ----------------------------------------------------
BYTES_PER_WEIGHT = {"q4_k": 144 / 256, "q6_k": 210 / 256, "fp8": 1 + 4 / 128**2, "nvfp4": 9 / 16, "q8g32": 34 / 32}


def work(case):
    kind = case["kind"]
    if kind in ("q8_mlp", "prefill_mlp"):
        m = case["m"]
        gate, down = (case["layout"], "q4_k") if kind == "prefill_mlp" else ("q4_k", "q6_k")
        weights = HIDDEN * FFN * (2 * BYTES_PER_WEIGHT[gate] + BYTES_PER_WEIGHT[down])
        return {"bytes": weights + 2 * HIDDEN + m * HIDDEN * 8, "flops": 6.0 * m * HIDDEN * FFN}
    m, n, k = case.get("m", 1), case["n"], case["k"]
    if kind == "q8_project":
        out, pair, layout = (8 if case["residual"] else 4), 1, case["quant"]
    else:
        out = {"bf16": 2, "swiglu": 2, "fp32": 4, "residual": 8}[case["epilogue"]]
        pair, layout = (2 if case["epilogue"] == "swiglu" else 1), case.get("layout", "fp8")
    return {"bytes": pair * n * k * BYTES_PER_WEIGHT[layout] + m * k * 2 + m * n * out, "flops": 2.0 * pair * m * n * k}


# ---- the same results in 64 bits ---------------------------------------------

def _bf16_operands(layout, parts):
    """The operand rows that a BF16-activation kernel multiplies."""
    if layout != "q4_k":
        return parts
    ds, dm, q = parts  # the code's affine in FP32, rounded to BF16
    return (ds[..., None] * q - dm[..., None]).float().bfloat16().double().view(q.shape[0], -1)


def _full_operands(layout, parts):
    if layout == "q4_k":
        return (parts[0][..., None] * parts[2] - parts[1][..., None]).view(parts[2].shape[0], -1)
    return (parts[0][..., None] * parts[1]).view(parts[1].shape[0], -1)


def _contract(x, layout, n, k, seed, salt, operands):
    y = torch.empty(x.shape[0], n, dtype=torch.float64, device="cuda")
    for r, _, parts in MAKERS[layout](_generator(seed, salt), n, k, True):
        w = operands(layout, parts)
        y[:, r:r + w.shape[0]] = x @ w.t()
    return y


def _q8(x):
    """Q8 groups of 32: a = peak / 127 and codes round(x / a), in FP32 as the format says."""
    x = x.view(x.shape[0], -1, 32)
    peak = x.abs().amax(-1, keepdim=True)
    a = torch.where(peak == 0, torch.ones_like(peak), (peak.double() / 127).float())
    z = (x.double() / a.double()).float().round().clamp(-127, 127)
    return (z.double() * a.double()).flatten(1)


def _fp8_rows(x):
    b = x.view(x.shape[0], -1, 128)
    peak = b.abs().amax(-1, keepdim=True)
    s = torch.where(peak == 0, torch.ones_like(peak), (peak.double() / 448).float().clamp(min=2.0**-126))
    return ((b.double() / s.double()).float().to(torch.float8_e4m3fn).double() * s.double()).flatten(1)


def _nvfp4_rows(x):
    s, c = _nvfp4_blocks(x.view(x.shape[0], -1, 16))
    return (s.view(torch.float8_e4m3fn).double()[..., None] * _e2m1_values(c)).flatten(1)


def _rms(case, seed):
    h = _tokens(seed, case["m"], HIDDEN).double()
    return ((1 + _gamma(seed).double()) * h / (h.square().mean(-1, keepdim=True) + EPS).sqrt()).bfloat16().float(), h


def _swiglu(g, u):
    return (g * torch.sigmoid(g) * u).bfloat16().float()


def exact(case, seed):
    kind = case["kind"]
    if kind == "q8_mlp":
        x, h = _rms(case, seed)
        x = _q8(x)
        v = _q8(_swiglu(*(_contract(x, "q4_k", FFN, HIDDEN, seed, i, _full_operands) for i in (1, 2))))
        return h + _contract(v, "q6_k", HIDDEN, FFN, seed, 3, _full_operands)
    if kind == "prefill_mlp":
        x, h = _rms(case, seed)
        x = _nvfp4_rows(x) if case["layout"] == "nvfp4" else x.double()
        v = _swiglu(*(_contract(x, case["layout"], FFN, HIDDEN, seed, i, _bf16_operands) for i in (1, 2)))
        return h + _contract(v.double(), "q4_k", HIDDEN, FFN, seed, 3, _bf16_operands)
    m, n, k = case.get("m", 1), case["n"], case["k"]
    x = _tokens(seed, m, k).bfloat16().float()
    if kind == "q8_project":
        y = _contract(_q8(x), case["quant"], n, k, seed, 1, _full_operands)
        return y + _residual(seed, m, n).double() if case["residual"] else y
    layout = case.get("layout", "fp8")
    x = _fp8_rows(x) if kind == "fp8_project" else x.double()
    y = _contract(x, layout, n, k, seed, 1, _bf16_operands)
    if case["epilogue"] == "swiglu":
        u = _contract(x, layout, n, k, seed, 2, _bf16_operands)
        return y * torch.sigmoid(y) * u
    return y + _residual(seed, m, n).double() if case["epilogue"] == "residual" else y


def tolerance(case):
    # Each about four times the largest distance from exact() over the listed cases.
    kind = case["kind"]
    if kind in ("q8_mlp", "prefill_mlp"):
        # FP32 sums feed BF16 roundings and 4- or 8-bit codes: a sum in another order moves single values
        return {"rel": 3e-4}
    if kind == "q8_project" or case["epilogue"] in ("fp32", "residual"):
        return {"rel": 2e-6}  # FP32 sums
    return {"rel": 6e-3}  # BF16 results

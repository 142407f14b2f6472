"""The work a model runner has this library do, as measured cases.

Every case calls the Python mirror of the operator surface
(``kraken_amd.Backend``): the projections of a decode step and of a prompt
(``gemm``, ``gemm_group``, ``gemm_accumulate``), the int8 rung, and the routed
expert layer (``router_softmax``, ``router_topk``, ``moe_dispatch``).  Norms,
attention and the activation function between a prompt's projections belong to
the caller's other kernels, so their results are inputs here.

Weights are N(0, 0.02), quantized here on the GPU into the GGUF block formats;
activations are N(0, 1).  A handle is made once per activation type and kept,
as a program does.
"""
import math

import torch

import kraken_amd as K

FORMATS = {"q4_k": K.Q4_K, "q5_k": K.Q5_K, "q6_k": K.Q6_K, "q8_0": K.Q8_0, "q4_0": K.Q4_0}
DEV = "cuda"


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # the smallest call: one projection of a small model's decode step
        # (2048 x 2048, the shape of the library's CPU reference figure)
        {"name": "proj_q8_0_2048", "kind": "proj", "fmt": "q8_0", "act": "f32", "rows": 1, "n_in": 2048, "n_out": 2048},
        # one token through four Llama-2-7B-shaped layers, grouped and fused as
        # an engine issues them
        {"name": "decode_q4_k", "kind": "layers", "fmt": "q4_k", "fmt2": "q4_k", "act": "f16", "hidden": 4096, "ff": 11008,
         "kv": 4096, "layers": 4},
        # the output head of a 128256-word vocabulary: decode, and a prompt's last row
        {"name": "head_q6_k", "kind": "proj", "fmt": "q6_k", "act": "f16", "rows": 1, "n_in": 4096, "n_out": 128256},
        # the feed-forward projections (Llama-3-8B shape) of 8 sequences
        # decoded together, and of a small batch of draft tokens checked at
        # once (mixed Q4_K / Q6_K, as Q4_K_M files hold it)
        {"name": "ffn_8_q4_k", "kind": "ffn", "fmt": "q4_k", "fmt2": "q4_k", "act": "f16", "rows": 8, "hidden": 4096, "ff": 14336},
        {"name": "ffn_37_q4_k_m", "kind": "ffn", "fmt": "q4_k", "fmt2": "q6_k", "act": "f32", "rows": 37, "hidden": 4096, "ff": 14336},
        # the same projections over a prompt: one of ragged length in Q5_K_M,
        # and the full 2048-token chunk in Q4_K
        {"name": "ffn_509_q5_k_m", "kind": "ffn", "fmt": "q5_k", "fmt2": "q6_k", "act": "f32", "rows": 509, "hidden": 4096, "ff": 14336},
        {"name": "ffn_2048_q4_k", "kind": "ffn", "fmt": "q4_k", "fmt2": "q4_k", "act": "f16", "rows": 2048, "hidden": 4096, "ff": 14336},
        # a prompt's up projection on the int8 rung (Q8_0 weights, Q8 activations)
        {"name": "int8_512_q8_0", "kind": "int8", "fmt": "q8_0", "act": "f32", "rows": 512, "n_in": 4096, "n_out": 14336},
        # one routed-expert layer of a 128-expert, top-8 model: one token, 16
        # tokens, and prompts, in the reference engine's f16 activations and in f32
        {"name": "moe_1_q4_k", "kind": "moe", "fmt": "q4_k", "fmt2": "q4_k", "act": "f16", "rows": 1, "hidden": 4096, "ff": 1536,
         "experts": 128, "top": 8},
        {"name": "moe_16_q4_k_m", "kind": "moe", "fmt": "q4_k", "fmt2": "q6_k", "act": "f32", "rows": 16, "hidden": 4096, "ff": 1536,
         "experts": 128, "top": 8},
        {"name": "moe_160_q4_k", "kind": "moe", "fmt": "q4_k", "fmt2": "q4_k", "act": "f16", "rows": 160, "hidden": 4096, "ff": 1536,
         "experts": 128, "top": 8},
        {"name": "moe_512_q4_k", "kind": "moe", "fmt": "q4_k", "fmt2": "q4_k", "act": "f32", "rows": 512, "hidden": 4096, "ff": 1536,
         "experts": 128, "top": 8},
    ]


def _log(rng, lo, hi, step=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["proj", "layers", "ffn", "ffn", "int8", "moe", "moe"])
    # one format throughout, or the mixed files' Q6_K in the down (and v) projections
    fmt = rng.choice(["q4_k", "q4_k", "q5_k", "q6_k", "q8_0", "q4_0"])
    fmt2 = "q6_k" if fmt in ("q4_k", "q5_k") and rng.random() < 0.5 else fmt
    act = rng.choice(["f16", "f32"])
    hidden = _log(rng, 1024, 5120, 256)
    if kind == "proj":   # any row count up to a prompt's; heads of odd vocabularies at one row
        rows = _log(rng, 1, 1024)
        n_out = _log(rng, 512, 128256) if rows == 1 else _log(rng, 512, 16384)
        return {"kind": kind, "fmt": fmt, "act": act, "rows": rows, "n_in": hidden, "n_out": n_out}
    if kind == "int8":
        return {"kind": kind, "fmt": rng.choice(["q8_0", "q4_k", "q6_k"]), "act": act, "rows": _log(rng, 32, 1024), "n_in": hidden,
                "n_out": _log(rng, 1024, 14336)}
    if kind == "layers":
        return {"kind": kind, "fmt": fmt, "fmt2": fmt2, "act": act, "hidden": hidden, "ff": _log(rng, 2048, 14336, 256),
                "kv": rng.choice([hidden, hidden // 4]), "layers": 4}
    if kind == "ffn":
        return {"kind": kind, "fmt": fmt, "fmt2": fmt2, "act": act, "rows": _log(rng, 2, 2048), "hidden": min(hidden, 4096),
                "ff": _log(rng, 2048, 14336, 256)}
    fmt = rng.choice(["q4_k", "q4_k", "q8_0"])
    return {"kind": kind, "fmt": fmt, "fmt2": rng.choice([fmt, "q6_k"]) if fmt == "q4_k" else fmt, "act": act, "rows": _log(rng, 1, 512),
            "hidden": min(hidden, 4096), "ff": _log(rng, 512, 2048, 256), "experts": rng.choice([32, 64, 128]),
            "top": rng.choice([2, 4, 8])}


# -------------------------------------------- GGUF blocks on the GPU (torch) --
def _pack_k(v, bits):
    """Per 256 values eight sub-blocks of scale and min over `bits`-bit codes: (d, dmin, the 12 scale bytes, codes)."""
    s = v.view(-1, 8, 32)
    top = (1 << bits) - 1
    mn = (-s.amin(2)).clamp_min(0)
    sc = (s.amax(2) + mn).clamp_min(1e-12) / top
    d, dm = (sc.amax(1, keepdim=True) / 63).half(), (mn.amax(1, keepdim=True) / 63).half()
    ls = (sc / d.float()).round().clamp(0, 63)
    lm = (mn / dm.float().clamp_min(1e-12)).round().clamp(0, 63)
    q = ((s + (dm.float() * lm)[..., None]) / (d.float() * ls).clamp_min(1e-12)[..., None]).round_().clamp_(0, top).to(torch.uint8)
    ls, lm = ls.to(torch.uint8), lm.to(torch.uint8)
    packed = torch.cat([ls[:, :4] | ((ls[:, 4:] >> 4) << 6), lm[:, :4] | ((lm[:, 4:] >> 4) << 6), (ls[:, 4:] & 15) | ((lm[:, 4:] & 15) << 4)], 1)
    return d, dm, packed, q


def _u8(t):
    return t.contiguous().view(torch.uint8)


def quantize(fmt, v):
    """GGUF bytes of the f32 values v, whole blocks in order."""
    if fmt == "q8_0":
        b = v.view(-1, 32)
        d = (b.abs().amax(1, keepdim=True) / 127).half()
        q = (b / d.float().clamp_min(1e-12)).round_().clamp_(-127, 127).to(torch.int8)
        out = torch.cat([_u8(d), _u8(q)], 1)
    elif fmt == "q4_0":
        b = v.view(-1, 32)
        d = (torch.gather(b, 1, b.abs().argmax(1, keepdim=True)) / -8).half()
        q = (b / d.float() + 8).round_().clamp_(0, 15).to(torch.uint8)
        out = torch.cat([_u8(d), q[:, :16] | (q[:, 16:] << 4)], 1)
    elif fmt in ("q4_k", "q5_k"):
        d, dm, packed, q = _pack_k(v, 4 if fmt == "q4_k" else 5)
        lo, high = q & 15, []
        if fmt == "q5_k":
            h = torch.zeros_like(q[:, 0])
            for c in range(8):
                h |= (q[:, c] >> 4) << c
            high = [h]
        out = torch.cat([_u8(d), _u8(dm), packed, *high, (lo[:, 0::2] | (lo[:, 1::2] << 4)).flatten(1)], 1)
    elif fmt == "q6_k":
        s = v.view(-1, 16, 16)
        sc = s.abs().amax(2).clamp_min(1e-12) / 31
        d = (sc.amax(1, keepdim=True) / 127).half()
        ls = (sc / d.float()).round().clamp(1, 127)
        q = ((s / (d.float() * ls)[..., None]).round_().clamp_(-32, 31) + 32).to(torch.uint8).view(-1, 2, 4, 32)
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2).flatten(1)
        qh = ((q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)).flatten(1)
        out = torch.cat([ql, qh, _u8(ls.to(torch.int8)), _u8(d)], 1)
    else:
        raise ValueError(fmt)
    return out.reshape(-1)


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def dequantize(fmt, raw, n_rows, n_in):
    """The blocks' values in 64 bits, [n_rows, n_in]."""
    if fmt == "q8_0":
        b = raw.view(-1, 34)
        v = _f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8)
    elif fmt == "q4_0":
        b = raw.view(-1, 18)
        v = _f16(b[:, :2]) * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    elif fmt in ("q4_k", "q5_k"):
        b = raw.view(-1, 144 if fmt == "q4_k" else 176)
        p = b[:, 4:16]
        sc = torch.cat([p[:, :4] & 63, (p[:, 8:] & 15) | ((p[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        if fmt == "q5_k":
            q = q | torch.stack([((b[:, 16:48] >> c) & 1) << 4 for c in range(8)], 1)
        v = (_f16(b[:, :2]) * sc)[..., None] * q - (_f16(b[:, 2:4]) * mn)[..., None]
    else:
        b = raw.view(-1, 210)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        q = torch.cat([ql & 15, ql >> 4], 2) | torch.cat([((qh >> (2 * j)) & 3) << 4 for j in range(4)], 2)
        ds = _f16(b[:, 208:]) * b[:, 192:208].contiguous().view(torch.int8)
        v = ds[..., None] * (q.view(-1, 16, 16).double() - 32)
    return v.reshape(n_rows, n_in)


def _weights(g, fmt, n_rows, n_in):
    parts, step = [], max(1, (1 << 26) // n_in)
    for r in range(0, n_rows, step):
        v = torch.randn(min(step, n_rows - r) * n_in, generator=g, device=DEV).mul_(0.02)
        parts.append(quantize(fmt, v))
    return torch.cat(parts) if len(parts) > 1 else parts[0]


# --------------------------------------------------------- prepare and run --
_handles = {}


def _handle(case):
    key = (case["act"], case["kind"] == "int8")
    if key not in _handles:
        _handles[key] = K.Backend(0, K.ACT_F16 if case["act"] == "f16" else K.ACT_F32)
        if key[1]:
            _handles[key].set_gemm_path(K.PATH_INT8)
    return _handles[key]


def _inputs(case, seed):
    """The case's tensors by name, from the seed alone; the same ones for prepare() and exact()."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)
    dt = torch.float16 if case["act"] == "f16" else torch.float32
    x = lambda *shape: torch.randn(*shape, generator=g, device=DEV).to(dt)  # noqa: E731
    kind, t = case["kind"], {}
    if kind in ("proj", "int8"):
        t["x"] = x(case["rows"], case["n_in"])
        t["w"] = _weights(g, case["fmt"], case["n_out"], case["n_in"])
    elif kind == "layers":
        t["h0"] = x(1, case["hidden"])
        t["layers"] = []
        for _ in range(case["layers"]):
            L = {"x1": x(1, case["hidden"]), "attn": x(1, case["hidden"]), "x2": x(1, case["hidden"])}
            for name, f, n_out, n_in in _layer_shapes(case):
                L[name] = _weights(g, f, n_out, n_in)
            t["layers"].append(L)
    elif kind == "ffn":
        t["x"], t["mid"] = x(case["rows"], case["hidden"]), x(case["rows"], case["ff"])
        for name, f, n_out, n_in in (("gate", "fmt", "ff", "hidden"), ("up", "fmt", "ff", "hidden"), ("down", "fmt2", "hidden", "ff")):
            t[name] = _weights(g, case[f], case[n_out], case[n_in])
    else:
        t["x"], t["logits"] = x(case["rows"], case["hidden"]), x(case["rows"], case["experts"])
        for name, f, n_out, n_in in _bank_shapes(case):
            t[name] = _weights(g, f, case["experts"] * n_out, n_in)
    return t


def _layer_shapes(c):
    h, ff, kv = c["hidden"], c["ff"], c["kv"]
    return [("q", c["fmt"], h, h), ("k", c["fmt"], kv, h), ("v", c["fmt2"], kv, h), ("o", c["fmt"], h, h), ("gate", c["fmt"], ff, h),
            ("up", c["fmt"], ff, h), ("down", c["fmt2"], h, ff)]


def _bank_shapes(c):
    return [("gate", c["fmt"], c["ff"], c["hidden"]), ("up", c["fmt"], c["ff"], c["hidden"]), ("down", c["fmt2"], c["hidden"], c["ff"])]


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], s["be"] = case, _handle(case)
    kind, dt = case["kind"], s["x" if "x" in s else "h0"].dtype
    new = lambda *shape, dtype=dt: torch.empty(*shape, dtype=dtype, device=DEV)  # noqa: E731
    if kind in ("proj", "int8"):
        s["out"] = new(case["rows"], case["n_out"])
    elif kind == "layers":
        s["h"] = new(1, case["hidden"])
        for L in s["layers"]:
            L["qkv"] = [new(1, case["hidden"]), new(1, case["kv"]), new(1, case["kv"])]
            L["act"] = [new(1, case["ff"]), new(1, case["ff"])]
    elif kind == "ffn":
        s["gu"] = [new(case["rows"], case["ff"]), new(case["rows"], case["ff"])]
        s["out"] = new(case["rows"], case["hidden"])
    else:
        n, e, k = case["rows"], case["experts"], case["top"]
        entries = []
        for i in range(e):
            en = K.MoeEntry()
            for m, (name, f, n_out, n_in) in enumerate(_bank_shapes(case)):
                rb = K.row_bytes(FORMATS[f], n_in)
                en.p[m], en.n_out[m], en.n_in[m] = s[name].data_ptr() + i * n_out * rb, n_out, n_in
                en.row_bytes[m], en.type[m], en.present[m] = rb, FORMATS[f], 1
            entries.append(en)
        s["table"] = torch.frombuffer(bytearray(K.moe_table_bytes(entries)), dtype=torch.uint8).to(DEV)
        s["be"].moe_table_forget(s["table"])   # an earlier model's table may have lain there
        s["probs"], s["ids"] = new(n, e, dtype=torch.float32), new(n, k, dtype=torch.int32)
        s["wts"], s["out"] = new(n, k, dtype=torch.float32), new(n, case["hidden"])
    return s


def run(s):
    c, be = s["case"], s["be"]
    kind = c["kind"]
    if kind in ("proj", "int8"):
        be.gemm(s["out"], s["x"], s["w"], FORMATS[c["fmt"]], c["n_out"], c["n_in"], c["rows"])
        return s["out"]
    f, f2 = FORMATS[c["fmt"]], FORMATS[c["fmt2"]]
    if kind == "layers":
        h, ff, kv = c["hidden"], c["ff"], c["kv"]
        s["h"].copy_(s["h0"])   # the token's embedding opens the residual stream
        for L in s["layers"]:
            be.gemm_group(L["qkv"], L["x1"], [L["q"], L["k"], L["v"]], f, [h, kv, kv], h, 1, wts=None if f == f2 else [f, f, f2])
            be.gemm_accumulate(s["h"], L["attn"], L["o"], f, h, h, 1)
            be.gemm_group(L["act"], L["x2"], [L["gate"], L["up"]], f, [ff, ff], h, 1, silu=True)
            be.gemm_accumulate(s["h"], L["act"][0], L["down"], f2, h, ff, 1)
        return {"qkv": [L["qkv"] for L in s["layers"]], "act": [L["act"][0] for L in s["layers"]], "h": s["h"]}
    if kind == "ffn":
        be.gemm_group(s["gu"], s["x"], [s["gate"], s["up"]], f, [c["ff"], c["ff"]], c["hidden"], c["rows"])
        be.gemm(s["out"], s["mid"], s["down"], f2, c["hidden"], c["ff"], c["rows"])
        return {"gate": s["gu"][0], "up": s["gu"][1], "down": s["out"]}
    n, e, k = c["rows"], c["experts"], c["top"]
    be.router_softmax(s["probs"], s["logits"], n, e)
    be.router_topk(s["probs"], n, e, k, s["ids"], s["wts"])
    be.moe_dispatch(s["table"], 0, e, s["ids"], s["wts"], s["x"], s["out"], n, c["hidden"], c["ff"], k)
    return {"probs": s["probs"], "ids": s["ids"], "wts": s["wts"], "out": s["out"]}


# ------------------------------------------------------- work and tolerance --
def work(case):
    a = 2 if case["act"] == "f16" else 4
    rb = lambda f, n: n // K.BLOCK_VALUES[FORMATS[f]] * K.BLOCK_BYTES[FORMATS[f]]  # noqa: E731
    kind, m = case["kind"], case.get("rows", 1)
    if kind in ("proj", "int8"):
        n, k = case["n_out"], case["n_in"]
        return {"bytes": n * rb(case["fmt"], k) + a * m * (n + k), "flops": 2 * m * n * k}
    if kind == "layers":
        by = sum(n_out * rb(f, n_in) + a * n_out for _, f, n_out, n_in in _layer_shapes(case)) + 3 * a * case["hidden"]
        return {"bytes": case["layers"] * by, "flops": case["layers"] * sum(2 * n_out * n_in for _, _, n_out, n_in in _layer_shapes(case))}
    mats = _bank_shapes(case)
    if kind == "ffn":
        return {"bytes": sum(n_out * rb(f, n_in) for _, f, n_out, n_in in mats) + a * m * (2 * case["hidden"] + 3 * case["ff"]),
                "flops": sum(2 * m * n_out * n_in for _, _, n_out, n_in in mats)}
    # experts that m tokens reach when each picks `top` of them at random
    e, k = case["experts"], case["top"]
    reached = e * (1 - (1 - k / e) ** m)
    return {"bytes": int(reached * sum(n_out * rb(f, n_in) for _, f, n_out, n_in in mats)) + a * m * (2 * case["hidden"] + e),
            "flops": sum(2 * m * k * n_out * n_in for _, _, n_out, n_in in mats)}


def tolerance(case):
    # About four times what each path is off the 64-bit result: 32-bit sums
    # of exact products (rows up to 8, small expert batches, the int8 rung),
    # one f16 rounding of each output (2.1e-4), f16 operands on the matrix
    # cores (2.9e-4), a decode layer's f16 residual stream (6e-4), the expert
    # layer's f16 rounding of each dot, mid row and partial sum (6.7e-4), and
    # its f16 operands for f32 batches of 32 tokens and more (5.1e-4).
    kind, f16, m = case["kind"], case["act"] == "f16", case.get("rows", 1)
    if kind == "moe":
        return {"rel": 2.7e-3} if f16 else {"rel": 2e-3} if m >= 32 else {"rel": 1e-5}
    if kind == "layers":
        return {"rel": 2.4e-3} if f16 else {"rel": 1e-5}
    if kind == "int8":
        return {"rel": 8e-4} if f16 else {"rel": 2e-6}
    if m > 8:
        return {"rel": 1.2e-3}
    return {"rel": 8e-4} if f16 else {"rel": 1e-5}


# -------------------------------------------------------- the 64-bit results --
def _dot(x, fmt, raw, n_out, n_in):
    x, out = x.double(), []
    step = max(1, (1 << 27) // n_in)
    per = raw.numel() // n_out
    for r in range(0, n_out, step):
        n = min(step, n_out - r)
        out.append(x @ dequantize(fmt, raw[r * per:(r + n) * per], n, n_in).t().contiguous())
    return torch.cat(out, 1)


def _silu(v):
    return v / (1 + torch.exp(-v))


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "int8":   # the rung's activations: int8 codes and one scale per 32 values
        b = t["x"].float().view(-1, 32)
        d = b.abs().amax(1, keepdim=True) / 127
        q = (b * torch.where(d > 0, 1 / d, 0 * d)).round()
        t["x"] = (q.double() * d.double()).view(case["rows"], case["n_in"])
    if kind in ("proj", "int8"):
        return _dot(t["x"], case["fmt"], t["w"], case["n_out"], case["n_in"])
    if kind == "layers":
        qkv, act, h = [], [], t["h0"].double()
        for L in t["layers"]:
            of = {name: (f, L[name], n_out, n_in) for name, f, n_out, n_in in _layer_shapes(case)}
            qkv.append([_dot(L["x1"], *of[name]) for name in ("q", "k", "v")])
            h = h + _dot(L["attn"], *of["o"])
            act.append(_silu(_dot(L["x2"], *of["gate"])) * _dot(L["x2"], *of["up"]))
            h = h + _dot(act[-1], *of["down"])
        return {"qkv": qkv, "act": act, "h": h}
    of = {name: (f, t[name], n_out, n_in) for name, f, n_out, n_in in _bank_shapes(case)}
    if kind == "ffn":
        return {"gate": _dot(t["x"], *of["gate"]), "up": _dot(t["x"], *of["up"]), "down": _dot(t["mid"], *of["down"])}
    p = torch.softmax(t["logits"].double(), 1)
    w, ids = torch.sort(p, dim=1, descending=True, stable=True)   # a tie keeps the lower id
    w, ids = w[:, :case["top"]], ids[:, :case["top"]]
    w = w / w.sum(1, keepdim=True)
    x, out = t["x"].double(), torch.zeros(case["rows"], case["hidden"], dtype=torch.float64, device=DEV)
    for e in range(case["experts"]):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if not tok.numel():
            continue
        one = lambda name, v: _dot(v, of[name][0], of[name][1].view(case["experts"], -1)[e], of[name][2], of[name][3])  # noqa: E731
        mid = _silu(one("gate", x[tok])) * one("up", x[tok])
        out.index_add_(0, tok, w[tok, slot][:, None] * one("down", mid))
    return {"probs": p, "ids": None, "wts": w, "out": out}

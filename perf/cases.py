"""The calls whose speed this framework is measured by.

Each case is one call of a program that keeps quantized weights on the GPU: the
matrix products of a decode step and of a prompt (`Context.matmul`,
`matmul_argmax`, `bind_matmul`), the GGML operators over stacked matrices
(`mul_mat`, `mul_mat_id`), the Llama decode step and the weight encoder.  The
shapes are those of a Llama-3-8B file (d 4096, FFN 14336, Q/K/V 6144, K or V
1024, vocabulary 128256), of a Mixtral FFN (8 experts of 14336x4096, top-2) and
of a Qwen2.5-0.5B FFN (4864x896).

Weights are GGUF blocks packed here from bell-shaped levels and scales of the
spread that N(0, 0.02) matrices have; activations are N(0, 1).
"""
import functools
import importlib

import torch

rlq = importlib.import_module("rust-llama_amd")
DT = rlq.DType

K_TYPES = ("Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K")
TYPES = ("Q8_0",) + K_TYPES

# Bounds of a drawn case, those of the largest listed ones.
MAX_FLOPS = 1.2e11
MAX_WEIGHTS = 128256 * 4096


def listed():
    return [
        # the smallest call: one token through the up projection of a 0.5B model
        {"name": "q8_0_4864x896_b1", "kind": "matmul", "type": "Q8_0", "rows": 4864, "cols": 896, "batch": 1},
        # one token, gate or up projection of an 8B model
        {"name": "q4_k_14336x4096_b1", "kind": "matmul", "type": "Q4_K", "rows": 14336, "cols": 4096, "batch": 1},
        # five sequences decoded together, down projection of an 8B model in a Q3_K file
        {"name": "q3_k_4096x14336_b5", "kind": "matmul", "type": "Q3_K", "rows": 4096, "cols": 14336, "batch": 5},
        # one token's logits and greedy choice: the output head
        {"name": "q6_k_128256x4096_b1_argmax", "kind": "argmax", "type": "Q6_K", "rows": 128256, "cols": 4096,
         "batch": 1},
        # thirty-two sequences decoded together, Q/K/V of an 8B model in a Q5_K file
        {"name": "q5_k_6144x4096_b32", "kind": "matmul", "type": "Q5_K", "rows": 6144, "cols": 4096, "batch": 32},
        # a short prompt through a K or V projection
        {"name": "q4_k_1024x4096_b77", "kind": "matmul", "type": "Q4_K", "rows": 1024, "cols": 4096, "batch": 77},
        # a prompt through a 0.5B model's up projection
        {"name": "q8_0_4864x896_b200", "kind": "matmul", "type": "Q8_0", "rows": 4864, "cols": 896, "batch": 200},
        # a full micro-batch of a prompt through gate or up of an 8B model
        {"name": "q4_k_14336x4096_b512", "kind": "matmul", "type": "Q4_K", "rows": 14336, "cols": 4096, "batch": 512},
        # a long prompt through the down projection, which a Q4_K_M file keeps in Q6_K
        {"name": "q6_k_4096x14336_b1000", "kind": "matmul", "type": "Q6_K", "rows": 4096, "cols": 14336,
         "batch": 1000},
        # a short prompt through the experts of a Mixtral FFN layer
        {"name": "moe_q4_k_8x14336x4096_t45", "kind": "mul_mat_id", "type": "Q4_K", "rows": 14336, "cols": 4096,
         "experts": 8, "slots": 2, "tokens": 45},
        # one decode step of the 8B layer shape in a Q4_K_M layout, at context 1000
        {"name": "llama_step_4x4096_ctx1000", "kind": "step", "type": "Q4_K", "more": "Q6_K", "width": 4096,
         "ffn": 14336, "layers": 4, "vocabulary": 128256, "context": 1000},
        # a weight matrix encoded for a GGUF file
        {"name": "encode_q4_k_4096x4096", "kind": "encode", "type": "Q4_K", "rows": 4096, "cols": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of lo..hi."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _cols(rng, t, lo, hi):
    return 32 * _log(rng, lo // 32, hi // 32) if t == "Q8_0" else 256 * _log(rng, max(1, lo // 256), hi // 256)


def _batch(rng):
    """One token, a few sequences, or a prompt or a large serving batch."""
    k = rng.random()
    return 1 if k < 0.25 else rng.randint(2, 8) if k < 0.5 else _log(rng, 9, 1024)


def draw(rng):
    kind = rng.choices(("matmul", "argmax", "mul_mat", "mul_mat_id", "step", "encode"), (60, 8, 8, 10, 8, 6))[0]
    t = rng.choice(TYPES)
    if kind in ("matmul", "argmax"):
        rows = _log(rng, 64, 32768) if kind == "matmul" else _log(rng, 4096, 131072)
        cols, batch = _cols(rng, t, 256, 14336), _batch(rng)
        while rows * cols > MAX_WEIGHTS:
            rows //= 2
        while 2.0 * rows * cols * batch > MAX_FLOPS:
            batch //= 2
        return {"kind": kind, "type": t, "rows": rows, "cols": cols, "batch": batch}
    if kind == "mul_mat":
        n2, share = rng.choice((1, 2, 4)), rng.choice((1, 2))
        return {"kind": kind, "type": t, "rows": _log(rng, 64, 8192), "cols": _cols(rng, t, 256, 4096), "n2": n2,
                "share": share, "ncols": _log(rng, 1, 128), "packed": rng.random() < 0.5}
    if kind == "mul_mat_id":
        rows, cols, experts = _log(rng, 512, 14336), _cols(rng, t, 512, 4096), rng.choice((4, 8, 16))
        return {"kind": kind, "type": t, "rows": rows, "cols": cols, "experts": experts, "slots": rng.choice((1, 2, 4)),
                "tokens": 1 if rng.random() < 0.4 else _log(rng, 2, 256)}
    if kind == "step":
        width = rng.choice((1024, 2048, 4096))
        return {"kind": kind, "type": rng.choice(("Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0")), "more": "Q6_K",
                "width": width, "ffn": 256 * _log(rng, width // 256, 56), "layers": rng.randint(1, 4),
                "vocabulary": 16 * _log(rng, 256, 8016), "context": _log(rng, 1, 1000)}
    return {"kind": kind, "type": t, "rows": _log(rng, 64, 4096), "cols": _cols(rng, t, 256, 4096)}


# ---- weights --------------------------------------------------------------------

def _levels(gen, n, lo, hi, sd, width=256):
    """[n, width] whole levels in lo..hi, normal about the middle."""
    x = torch.randn((n, width), generator=gen, device="cuda", dtype=torch.float32)
    return x.mul_(sd).add_((lo + hi) / 2).round_().clamp_(lo, hi).to(torch.int16)


def _ints(gen, n, lo, hi, width):
    return torch.randint(lo, hi + 1, (n, width), generator=gen, device="cuda", dtype=torch.int16)


def _half(gen, n, middle):
    """[n, 1] f16 super-scales of 0.75 to 1.25 times `middle`."""
    u = torch.rand((n, 1), generator=gen, device="cuda", dtype=torch.float32)
    return (u * 0.5 + 0.75).mul_(middle).to(torch.float16)


def _bytes(*parts):
    """GGUF blocks from their fields in order: u8 values in whole numbers, or f16."""
    return torch.cat([p.view(torch.uint8) if p.dtype == torch.float16 else (p & 255).to(torch.uint8) for p in parts],
                     dim=1)


def _two_bits(q):
    """Levels 0..3 of 256 values -> 64 bytes: value 128h + 32s + j in bits 2s of byte 32h + j."""
    q = q.view(-1, 2, 4, 32)
    return (q[:, :, 0] | q[:, :, 1] << 2 | q[:, :, 2] << 4 | q[:, :, 3] << 6).reshape(-1, 64)


def _nibbles(q):
    """Levels 0..15 of 256 values -> 128 bytes: value 64g + j low, 64g + 32 + j high in byte 32g + j."""
    q = q.view(-1, 4, 2, 32)
    return (q[:, :, 0] | q[:, :, 1] << 4).reshape(-1, 128)


def _six_bit_pairs(sc, mn):
    """The 12 bytes of eight 6-bit scales and minima."""
    low, high = sc[:, :4] | (sc[:, 4:] >> 4) << 6, mn[:, :4] | (mn[:, 4:] >> 4) << 6
    return torch.cat([low, high, (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], dim=1)


def _each(x, n):
    return x.repeat_interleave(n, dim=1)


def make_blocks(t, n, gen, values=False):
    """n GGUF blocks of type t and, if asked, the values they stand for, in 64 bits."""
    f64 = torch.float64
    if t == "Q8_0":
        q, d = _levels(gen, n, -127, 127, 42.0, 32), _half(gen, n, 0.02 / 42)
        return _bytes(d, q), d.to(f64) * q if values else None
    if t in ("Q4_K", "Q5_K"):
        top = 15 if t == "Q4_K" else 31
        q, sc = _levels(gen, n, 0, top, top / 4.4), _ints(gen, n, 20, 63, 8)
        mn = (sc.float() * (top / (top + 1.0))).round().to(torch.int16)
        d = _half(gen, n, 0.02 / (41.5 * top / 4.4))
        dmin = (d.float() * ((top + 1) / 2)).to(torch.float16)
        head = [d, dmin, _six_bit_pairs(sc, mn)]
        if t == "Q5_K":
            b = (q >> 4).view(-1, 8, 32)
            head.append(sum(b[:, s] << s for s in range(8)))
        w = d.to(f64) * (_each(sc, 32) * q) - dmin.to(f64) * _each(mn, 32) if values else None
        return _bytes(*head, _nibbles(q & 15)), w
    if t == "Q6_K":
        q, d = _levels(gen, n, -32, 31, 13.0), _half(gen, n, 0.02 / (13 * 98))
        sc = _ints(gen, n, 70, 127, 16) * (_ints(gen, n, 0, 1, 16) * 2 - 1)
        sc[:, 0] = -128
        u = (q + 32).view(-1, 2, 4, 32)
        ql = torch.stack([u[:, :, 0] & 15 | (u[:, :, 2] & 15) << 4, u[:, :, 1] & 15 | (u[:, :, 3] & 15) << 4], dim=2)
        qh = _two_bits((u >> 4).reshape(-1, 256))
        return _bytes(ql.reshape(-1, 128), qh, sc, d), d.to(f64) * (_each(sc, 16) * q) if values else None
    if t == "Q3_K":
        q, d = _levels(gen, n, -4, 3, 1.7), _half(gen, n, 0.02 / (1.7 * 24))
        sc = _ints(gen, n, 16, 31, 16) * (_ints(gen, n, 0, 1, 16) * 2 - 1)
        u, s = q + 4, sc + 32
        h = (u >> 2).view(-1, 8, 32)
        hmask = sum(h[:, k] << k for k in range(8))
        top = (s >> 4).view(-1, 4, 4)
        scales = torch.cat([s[:, :8] & 15 | (s[:, 8:] & 15) << 4,
                            top[:, 0] | top[:, 1] << 2 | top[:, 2] << 4 | top[:, 3] << 6], dim=1)
        return _bytes(hmask, _two_bits(u & 3), scales, d), d.to(f64) * (_each(sc, 16) * q) if values else None
    q, sc = _levels(gen, n, 0, 3, 0.9), _ints(gen, n, 7, 15, 16)  # Q2_K
    d = _half(gen, n, 0.02 / (0.9 * 11))
    dmin = (d.float() * 1.5).to(torch.float16)
    w = d.to(f64) * (_each(sc, 16) * q) - dmin.to(f64) * _each(sc, 16) if values else None
    return _bytes(sc | sc << 4, _two_bits(q), d, dmin), w


def _per_block(t):
    return 32 if t == "Q8_0" else 256


def make_matrix(t, rows, cols, gen, values=False):
    b, w = make_blocks(t, rows * cols // _per_block(t), gen, values)
    return b.reshape(-1), w.reshape(rows, cols) if values else None


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


# ---- what the products compute, in 64 bits --------------------------------------

def quantized(t, x):
    """The activations as the product with weights of type t sees them: rounded
    to Q8_0 or Q8_K as the formats define it (each f32 step rounded once)."""
    f32, f64 = torch.float32, torch.float64
    b = x.reshape(-1, _per_block(t)).to(f64)
    if t == "Q8_0":
        d = (b.abs().amax(1, keepdim=True) / 127).to(f32)
        v = (b * (1 / d.to(f64)).to(f32).to(f64)).to(f32).to(f64)
        q, d = v.sign() * (v.abs() + 0.5).floor(), d.to(torch.float16)
    else:
        inverse = (-127 / b.gather(1, b.abs().argmax(1, keepdim=True))).to(f32).to(f64)
        q, d = (b * inverse).to(f32).to(f64).round(), (1 / inverse).to(f32)
    return (q * d.to(f64)).reshape(x.shape)


# ---- the protocol -------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _context():
    return rlq.Context(0)


def _inputs(case, seed, values=False):
    """Weight bytes (with `values` their values) and activations of a product."""
    gen, t = _generator(seed), case["type"]
    mats = case.get("experts") or case.get("n2") or 1
    data, w = make_matrix(t, mats * case["rows"], case["cols"], gen, values)
    if case["kind"] == "mul_mat_id":
        x = _normal(gen, case["tokens"], 1, case["cols"])
    elif case["kind"] == "mul_mat":
        x = _normal(gen, 1, case["n2"] * case["share"], case["ncols"], case["cols"])
    else:
        x = _normal(gen, case["batch"], case["cols"])
    ids = None
    if case["kind"] == "mul_mat_id":  # distinct experts of each token
        chance = torch.rand((case["tokens"], mats), generator=gen, device="cuda")
        ids = chance.argsort(dim=1)[:, :case["slots"]].to(torch.int32).contiguous()
    return data, w, x, ids


def _prepare_step(case, seed):
    gen, W, F, V = _generator(seed), case["width"], case["ffn"], case["vocabulary"]
    heads, kv = W // 128, max(1, W // 512)
    base, more = case["type"], case["more"]
    layers = []
    for i in range(case["layers"]):
        # as a Q4_K_M file does, the value and down matrices of some layers in the larger type
        vd = more if i % 2 == 0 else base
        shapes = {"query": (base, W, W), "key": (base, kv * 128, W), "value": (vd, kv * 128, W),
                  "attention_output": (base, W, W), "gate": (base, F, W), "up": (base, F, W), "down": (vd, W, F)}
        layer = {k: make_matrix(*s, gen)[0] for k, s in shapes.items()}
        layer.update({k: _normal(gen, W) * 0.05 + 1.0 for k in ("attention_norm", "feed_forward_norm")})
        layer["types"] = {k: int(DT[s[0]]) for k, s in shapes.items()}
        layers.append(layer)
    emb = make_matrix("Q4_K", V, W, gen)[0].view(-1, 144)
    emb[:, :4] = (emb[:, :4].contiguous().view(torch.float16) * 50.0).view(torch.uint8)  # rows of spread 1
    tensors = {"embedding": emb.reshape(-1), "output_norm": _normal(gen, W) * 0.05 + 1.0,
               "output": make_matrix("Q6_K", V, W, gen)[0], "layers": layers}
    cfg = rlq.LlamaConfig(V, W, F, heads, kv, 1024, case["layers"], 1e-5, 500000.0, 0.0, DT[base], DT.Q6_K, DT.Q4_K)
    ctx = _context()
    model = rlq.LlamaModel(ctx, cfg, tensors)
    del tensors, layers, emb
    tokens = torch.randint(0, V, (case["context"] + 1,), generator=gen, device="cuda").tolist()
    hidden = torch.empty(W, dtype=torch.float32, device="cuda")
    for pos in range(case["context"]):
        model.embedding(tokens[pos], hidden)
        model.step(hidden, pos, embedding=False, logits=False)
    ctx.sync()
    return {"model": model, "token": tokens[-1], "pos": case["context"], "hidden": hidden}


def prepare(case, seed):
    kind, ctx = case["kind"], _context()
    if kind == "step":
        return dict(_prepare_step(case, seed), kind=kind)
    if kind == "encode":
        return {"kind": kind, "type": DT[case["type"]], "x": _normal(_generator(seed), case["rows"], case["cols"]) * 0.02}
    data, _, x, ids = _inputs(case, seed)
    mats = case.get("experts") or case.get("n2") or 1
    w = rlq.Weights(ctx, DT[case["type"]], data, case["rows"], case["cols"], mats)
    s = {"kind": kind, "w": w, "x": x, "ids": ids, "x_dtype": DT.F32}
    if kind == "mul_mat" and case["packed"]:
        s["x_dtype"] = rlq.matvec_activation_dtype(DT[case["type"]])
        s["x"] = ctx.quantize(s["x_dtype"], x.reshape(-1, case["cols"])).reshape(*x.shape[:3], -1)
        ctx.sync()
    if kind in ("matmul", "argmax") and case["batch"] <= 8:  # a serving loop: its buffers are bound once
        s["y"] = torch.empty((case["batch"], case["rows"]), dtype=torch.float32, device="cuda")
        s["best"] = torch.empty(case["batch"], dtype=torch.int32, device="cuda") if kind == "argmax" else None
        s["call"] = ctx.bind_matmul(w, x, s["y"], s["best"])
    return s


def run(s):
    kind, ctx = s["kind"], _context()
    if kind == "step":
        model = s["model"]
        model.truncate(s["pos"])
        model.embedding(s["token"], s["hidden"])
        _, logits, best = model.step(s["hidden"], s["pos"], embedding=False, argmax=True)
        return {"hidden": s["hidden"], "logits": logits, "best": best}
    if kind == "encode":
        return ctx.quantize(s["type"], s["x"])
    if "call" in s:
        s["call"]()
        return s["y"] if s["best"] is None else {"y": s["y"], "best": s["best"]}
    if kind == "matmul":
        return ctx.matmul(s["w"], s["x"])
    if kind == "argmax":
        y, best = ctx.matmul_argmax(s["w"], s["x"])
        return {"y": y, "best": best}
    if kind == "mul_mat":
        return ctx.mul_mat(s["w"], s["x"], s["x_dtype"])
    return ctx.mul_mat_id(s["w"], s["x"], s["ids"])


def _row_bytes(t, cols):
    return rlq.row_bytes(DT[t], cols)


def work(case):
    kind, t = case["kind"], case["type"]
    if kind == "step":
        W, F, V, L = case["width"], case["ffn"], case["vocabulary"], case["layers"]
        kvw, more = max(1, W // 512) * 128, (L + 1) // 2
        same = L * (_row_bytes(t, W) * (2 * W + kvw + 2 * F))
        vd = more * (_row_bytes(case["more"], W) * kvw + _row_bytes(case["more"], F) * W) \
            + (L - more) * (_row_bytes(t, W) * kvw + _row_bytes(t, F) * W)
        params = L * (2 * W * W + 2 * W * kvw + 3 * W * F) + V * W
        rows = case["context"] + 1
        return {"bytes": same + vd + _row_bytes("Q6_K", W) * V + 8 * L * rows * kvw + 4 * V,
                "flops": 2 * params + 4 * L * rows * W}
    rows, cols = case["rows"], case["cols"]
    if kind == "encode":
        return {"bytes": rows * (4 * cols + _row_bytes(t, cols)), "flops": 0}
    if kind == "mul_mat_id":
        pairs = case["tokens"] * case["slots"]
        mats, columns = min(case["experts"], pairs), case["tokens"]
    elif kind == "mul_mat":
        mats, columns = case["n2"], case["n2"] * case["share"] * case["ncols"]
        pairs = columns
    else:
        mats, columns = 1, case["batch"]
        pairs = columns
    x = columns * (rlq.row_bytes(rlq.matvec_activation_dtype(DT[t]), cols) if case.get("packed") else 4 * cols)
    return {"bytes": mats * rows * _row_bytes(t, cols) + x + 4 * pairs * rows, "flops": 2.0 * pairs * rows * cols}


def tolerance(case):
    kind = case["kind"]
    if kind in ("encode", "step"):
        # bytes; and a step promises the f32 results of one fixed order of operations bit for bit (a
        # single last bit of its input moves the logits by 2e-2: every layer rounds to 8 bits again)
        return "exact"
    # exact block integers and f32 sums of 1 to 448 block terms: 0.5e-7 to 3.1e-7 from 64 bits
    return {"rel": 1.2e-6, "max": 2e-5, "differ": 0.01}


def exact(case, seed):
    kind, t = case["kind"], case["type"]
    if kind in ("step", "encode"):
        # bytes; and a chain of 8-bit roundings, which 64 bits would round to other levels
        return None
    _, w, x, ids = _inputs(case, seed, values=True)
    a = quantized(t, x)
    if kind == "mul_mat_id":
        w, a = w.view(case["experts"], case["rows"], case["cols"]), a[:, 0]
        y = torch.empty((*ids.shape, case["rows"]), dtype=torch.float64, device="cuda")
        for e in range(case["experts"]):
            at = (ids == e).nonzero(as_tuple=True)
            y[at] = a[at[0]] @ w[e].t()
        return y
    if kind == "mul_mat":
        w = w.view(case["n2"], case["rows"], case["cols"])
        return torch.stack([a[0, i] @ w[i // case["share"]].t() for i in range(a.shape[1])]).unsqueeze(0)
    y = a @ w.t()
    return y if kind == "matmul" else {"y": y, "best": None}

"""The measured cases of this library: the quantized products of a GGUF
model's layers, each as a program calls them through swarmllm_amd.

Kinds (a case's "kind"):
  linear  one weight against a batch of rows (QMatMul.forward);
  layer   a decoder layer's weight products: q/k/v against one activation
          (QMatMul.forward_shared), the attention output, gate + up with the
          SiLU gate between them (forward_glu) and down. Every product gets
          an input of its own, so each is held to its own error and none
          carries another's rounding on;
  decode  the same for a stack of layers at one row, captured once as a HIP
          graph and replayed per token, as a serving loop runs it (eager
          calls at one row are bound by the host);
  moe     a mixture-of-experts layer's two grouped products: gate_up per
          token, down per (token, expert) pair with the router's weights
          (moe_forward; past 8 tokens the prompt form, moe_uses_prompt_kernel);
  wire    hidden states to the Q8_0 bytes peers exchange, and back.

Weights are GGUF blocks of N(0, 0.02) values, made here from the seed (a
plain quantizer per format, not the search that model files are made with:
the products do not depend on how the codes were chosen). Activations are
N(0, 1) with 1% of the channels 20 times larger, as hidden states have them.
"""
import math

import torch

import swarmllm_amd as sa
from swarmllm_amd import quant

DEV = "cuda"
# format: (ggml type, values a block, bytes a block)
FORMATS = {"q8_0": (8, 32, 34), "q4_k": (12, 256, 144), "q6_k": (14, 256, 210), "iq4_nl": (20, 32, 18),
           "mxfp4": (39, 32, 17)}
IQ4_NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
E2M1_DOUBLED = (0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12)
CHUNK = 1 << 25  # values quantized or dequantized at a time


def listed():
    return [
        # the smallest call: one token against one 4096-wide Q8_0 projection
        {"name": "linear_q8_0_1row", "kind": "linear", "fmt": "q8_0", "n": 4096, "k": 4096, "rows": 1},
        # the output head of a 128K vocabulary for one token: the longest stream of one weight
        {"name": "head_q6_k_1row", "kind": "linear", "fmt": "q6_k", "n": 128256, "k": 4096, "rows": 1},
        # a token through layers of an 8B model (Q4_K, Q6_K down): single-stream decode
        {"name": "decode_8b_1row", "kind": "decode", "fmt": "q4_k", "down": "q6_k", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "rows": 1, "layers": 2},
        # eight sequences decoded together through a 70B model's layer
        {"name": "batch_70b_8rows", "kind": "layer", "fmt": "q4_k", "down": "q6_k", "hidden": 8192, "kv": 1024,
         "ffn": 28672, "rows": 8},
        # an odd batch past one matrix-core tile: many sequences, or a speculated draft checked
        {"name": "batch_8b_21rows", "kind": "layer", "fmt": "q4_k", "down": "q6_k", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "rows": 21},
        # a short question
        {"name": "prompt_8b_77rows", "kind": "layer", "fmt": "q4_k", "down": "q6_k", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "rows": 77},
        # a prompt chunk
        {"name": "prompt_8b_512rows", "kind": "layer", "fmt": "q4_k", "down": "q6_k", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "rows": 512},
        # a long prompt in one call, the largest products
        {"name": "prompt_8b_2000rows", "kind": "layer", "fmt": "q4_k", "down": "q6_k", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "rows": 2000},
        # a prompt chunk of a model kept in Q8_0
        {"name": "prompt_q8_0_512rows", "kind": "layer", "fmt": "q8_0", "down": "q8_0", "hidden": 4096, "kv": 1024,
         "ffn": 14336, "rows": 512},
        # eight tokens of a 32-expert MXFP4 model, four experts each
        {"name": "moe_mxfp4_8tokens", "kind": "moe", "fmt": "mxfp4", "down": "mxfp4", "experts": 32, "topk": 4,
         "hidden": 2880, "width": 2880, "tokens": 8},
        # a prompt chunk of a 128-expert K-quant model, eight experts a token
        {"name": "moe_k_512tokens", "kind": "moe", "fmt": "q4_k", "down": "q6_k", "experts": 128, "topk": 8,
         "hidden": 2048, "width": 768, "tokens": 512},
        # a prompt's hidden states sent from one peer to the next
        {"name": "wire_2048x8192", "kind": "wire", "rows": 2048, "hidden": 8192},
    ]


LARGEST = 2000 * 218_103_808  # rows x weights of the largest listed case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "layer", "layer", "decode", "moe", "moe", "wire"])
    if kind == "linear":
        fmt = rng.choice(list(FORMATS))
        unit = FORMATS[fmt][1]
        k = unit * max(1, _log(rng, 512, 16384) // unit)
        n = _log(rng, 128, 131072 if k <= 4096 else 28672)
        rows = _log(rng, 1, 2048)
        return {"kind": kind, "fmt": fmt, "n": n, "k": k, "rows": max(1, min(rows, LARGEST // (n * k)))}
    if kind in ("layer", "decode"):
        fmt, down = rng.choice([("q4_k", "q6_k")] * 4 + [("q4_k", "q4_k"), ("q8_0", "q8_0"), ("iq4_nl", "iq4_nl")])
        hidden = 256 * rng.randint(4, 32)
        kv = 128 * rng.randint(1, max(1, hidden // 512))
        ffn = 256 * rng.randint(hidden // 256, 7 * hidden // 512)
        weights = hidden * (2 * hidden + 2 * kv + 3 * ffn)
        rows = min(_log(rng, 2, 2048), LARGEST // weights)
        if fmt not in ("q4_k",):
            rows = min(rows, 512)
        if kind == "decode":
            return {"kind": kind, "fmt": fmt, "down": down, "hidden": hidden, "kv": kv, "ffn": ffn,
                    "rows": rng.choice([1, 1, 2]), "layers": rng.randint(1, 3)}
        return {"kind": kind, "fmt": fmt, "down": down, "hidden": hidden, "kv": kv, "ffn": ffn, "rows": rows}
    if kind == "moe":
        fmt, down, unit = rng.choice([("mxfp4", "mxfp4", 32), ("q4_k", "q6_k", 256), ("q8_0", "q8_0", 32)])
        return {"kind": kind, "fmt": fmt, "down": down, "experts": rng.choice([8, 32, 60, 128]),
                "topk": rng.choice([2, 4, 8]), "hidden": unit * (rng.randint(1024, 3072) // unit),
                "width": unit * (rng.randint(512, 2880) // unit), "tokens": _log(rng, 1, 700)}
    return {"kind": kind, "rows": _log(rng, 1, 2048), "hidden": rng.choice([896, 2880, 4096, 5120, 8192])}


# ---- weights: GGUF blocks from values, and back in 64 bits -----------------


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape[:-1], -1)


def _pack_q8_0(x):
    b = x.view(-1, 32)
    d = (b.abs().amax(1, keepdim=True) / 127).to(torch.float16)
    q = torch.round(b / d.float().clamp_min(1e-8)).clamp(-127, 127).to(torch.int8)
    return torch.cat([_half_bytes(d), q.view(torch.uint8)], 1)


def _nearest(v, table):
    """Index of the nearest value of `table` (code order) to each of v."""
    t = torch.tensor(table, dtype=torch.float32, device=v.device)
    s, order = torch.sort(t)
    return order[torch.bucketize(v, (s[1:] + s[:-1]) / 2)].to(torch.uint8)


def _pack_iq4_nl(x):
    b = x.view(-1, 32)
    d = (b.abs().amax(1, keepdim=True) / 113).to(torch.float16)
    q = _nearest(b / d.float().clamp_min(1e-8), IQ4_NL)
    return torch.cat([_half_bytes(d), q[:, :16] | (q[:, 16:] << 4)], 1)


def _pack_mxfp4(x):
    b = x.view(-1, 32)
    e = torch.floor(torch.log2(b.abs().amax(1, keepdim=True).clamp_min(1e-30))) - 2 + 127
    q = _nearest(b * torch.exp2(128 - e), E2M1_DOUBLED)
    return torch.cat([e.to(torch.uint8), q[:, :16] | (q[:, 16:] << 4)], 1)


def _pack_q4_k(x):
    b = x.view(-1, 8, 32)
    low = (-b.amin(2)).clamp_min(0)
    step = (b.amax(2) + low) / 15
    d, dmin = (step.amax(1, keepdim=True) / 63).half(), (low.amax(1, keepdim=True) / 63).half()
    sc = torch.round(step / d.float().clamp_min(1e-8)).clamp(1, 63)
    mn = torch.round(low / dmin.float().clamp_min(1e-8)).clamp(0, 63)
    q = (b + (dmin.float() * mn)[:, :, None]) / (d.float() * sc)[:, :, None].clamp_min(1e-9)
    q = torch.round(q).clamp(0, 15).to(torch.uint8).view(-1, 4, 2, 32)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    return torch.cat([_half_bytes(d), _half_bytes(dmin), sc[:, :4] | ((sc[:, 4:] >> 4) << 6),
                      mn[:, :4] | ((mn[:, 4:] >> 4) << 6), (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4),
                      (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)], 1)


def _pack_q6_k(x):
    b = x.view(-1, 16, 16)
    step = b.abs().amax(2) / 31
    d = (step.amax(1, keepdim=True) / 127).half()
    sc = torch.round(step / d.float().clamp_min(1e-9)).clamp(1, 127)
    q = torch.round(b / (d.float() * sc)[:, :, None].clamp_min(1e-9)).clamp(-32, 31) + 32
    q = q.to(torch.uint8).view(-1, 2, 4, 32)  # half, group of 32, value
    ql = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _half_bytes(d)], 1)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _values(fmt, raw):
    """The values of GGUF blocks (uint8, flat) in float64."""
    b = raw.view(-1, FORMATS[fmt][2])
    if fmt == "q8_0":
        return (_half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if fmt in ("iq4_nl", "mxfp4"):
        head = 2 if fmt == "iq4_nl" else 1
        table = torch.tensor(IQ4_NL if head == 2 else E2M1_DOUBLED, dtype=torch.float64, device=raw.device)
        d = _half(b[:, :2]) if head == 2 else torch.exp2(b[:, :1].double() - 128)
        q = torch.cat([b[:, head:] & 15, b[:, head:] >> 4], 1)
        return (d * table[q.long()]).reshape(-1)
    if fmt == "q4_k":
        d, dmin, s = _half(b[:, 0:2]), _half(b[:, 2:4]), b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        return (q * (d * sc.double())[:, :, None] - (dmin * mn.double())[:, :, None]).reshape(-1)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    q = [(ql[:, :, g & 1] >> (4 * (g >> 1))) & 15 | (((qh >> (2 * g)) & 3) << 4) for g in range(4)]
    q = torch.stack(q, 2).reshape(-1, 16, 16).double() - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return (q * (_half(b[:, 208:210]) * sc)[:, :, None]).reshape(-1)


def _blocks(fmt, n, k, gen):
    """GGUF bytes (uint8 on the device) of an n x k weight of N(0, 0.02) values."""
    pack = globals()["_pack_" + fmt]
    step = max(1, CHUNK // k)
    parts = [pack(torch.randn((min(step, n - i), k), generator=gen, device=DEV) * 0.02).reshape(-1)
             for i in range(0, n, step)]
    return parts[0] if len(parts) == 1 else torch.cat(parts)


def _weight(fmt, shape, gen):
    """(format, shape, GGUF bytes) of a weight or a stack of weights."""
    return fmt, shape, _blocks(fmt, math.prod(shape[:-1]), shape[-1], gen)


def _qtensor(fmt, shape, raw):
    return sa.QTensor(raw, shape, sa.GgmlDType(FORMATS[fmt][0]))


def _acts(rows, k, gen):
    x = torch.randn((rows, k), generator=gen, device=DEV)
    return x * torch.where(torch.rand((k,), generator=gen, device=DEV) < 0.01, 20.0, 1.0)


# ---- the cases --------------------------------------------------------------


def _layer_shapes(c):
    """(name, format, n, k) of a layer's seven weights."""
    h, kv, f = c["hidden"], c["kv"], c["ffn"]
    return [("q", c["fmt"], h, h), ("k", c["fmt"], kv, h), ("v", c["fmt"], kv, h), ("o", c["fmt"], h, h),
            ("gate", c["fmt"], f, h), ("up", c["fmt"], f, h), ("down", c["down"], h, f)]


def _layer_acts(c, gen):
    return {name: _acts(c["rows"], k, gen)
            for name, k in (("qkv", c["hidden"]), ("o", c["hidden"]), ("mlp", c["hidden"]), ("down", c["ffn"]))}


def _layer_pass(w, x):
    q, k, v = sa.QMatMul.forward_shared(x["qkv"], [w["q"], w["k"], w["v"]])
    return [q, k, v, w["o"].forward(x["o"]), sa.forward_glu(x["mlp"], w["gate"], w["up"], "silu"),
            w["down"].forward(x["down"])]


def _routing(c, gen):
    """Each token's top-k distinct experts, the router's weights, and the
    pairs sorted by expert as the grouped products read them."""
    e, topk, tokens = c["experts"], c["topk"], c["tokens"]
    logits = torch.randn((tokens, e), generator=gen, device=DEV)
    top, experts = torch.topk(logits, topk, dim=1)
    expert_ids, sorted_ids = torch.sort(experts.reshape(-1), stable=True)
    return (sorted_ids.to(torch.int32), expert_ids.to(torch.int32),
            torch.softmax(top, 1).reshape(-1).contiguous(), experts)


def _seeded(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _inputs(c, seed):
    """(weights by name, inputs by name) of a case."""
    gen = _seeded(seed)
    kind = c["kind"]
    if kind == "linear":
        return {"w": _weight(c["fmt"], (c["n"], c["k"]), gen)}, {"x": _acts(c["rows"], c["k"], gen)}
    if kind == "layer":
        return {m: _weight(f, (n, k), gen) for m, f, n, k in _layer_shapes(c)}, _layer_acts(c, gen)
    if kind == "decode":
        return ({"%s%d" % (m, i): _weight(f, (n, k), gen) for i in range(c["layers"])
                 for m, f, n, k in _layer_shapes(c)}, [_layer_acts(c, gen) for _ in range(c["layers"])])
    if kind == "moe":
        e, h, f = c["experts"], c["hidden"], c["width"]
        w = {"gate_up": _weight(c["fmt"], (e, 2 * f, h), gen), "down": _weight(c["down"], (e, h, f), gen)}
        ids, eids, topw, experts = _routing(c, gen)
        return w, {"x": _acts(c["tokens"], h, gen), "y": _acts(c["tokens"] * c["topk"], f, gen), "ids": ids,
                   "eids": eids, "topw": topw, "experts": experts}
    return {}, {"x": _acts(c["rows"], c["hidden"], gen)}


def prepare(c, seed):
    w, x = _inputs(c, seed)
    w = {m: _qtensor(*t) for m, t in w.items()}
    s = {"kind": c["kind"], "x": x, "case": dict(c)}
    if c["kind"] == "moe":
        # one workspace a layer, kept by the program that runs it
        s.update(w=w, ws=sa.qtensor.Workspace(), prompt=sa.moe_uses_prompt_kernel(c["tokens"]))
        return s
    s["w"] = {m: sa.QMatMul.from_qtensor(t) for m, t in w.items()}
    if c["kind"] == "decode":
        for f in {c["fmt"], c["down"]}:
            sa.prepare(sa.GgmlDType(FORMATS[f][0]))
        layers = [{m: s["w"]["%s%d" % (m, i)] for m, *_ in _layer_shapes(c)} for i in range(c["layers"])]
        s["graph"] = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(s["graph"]):
            s["out"] = [_layer_pass(wl, xl) for wl, xl in zip(layers, x)]
    return s


def run(s):
    c, x, w = s["case"], s["x"], s.get("w")
    if s["kind"] == "linear":
        return w["w"].forward(x["x"])
    if s["kind"] == "layer":
        return _layer_pass(w, x)
    if s["kind"] == "decode":
        s["graph"].replay()
        return s["out"]
    if s["kind"] == "moe":
        up = sa.moe_forward(x["x"], w["gate_up"], x["ids"], x["eids"], None, c["topk"], s["prompt"], s["ws"])
        down = sa.moe_forward(x["y"], w["down"], x["ids"], x["eids"], x["topw"], c["topk"], s["prompt"], s["ws"])
        return [up, down]
    sent = quant.quantize_q8_0(x["x"])
    return [sent, quant.dequantize_q8_0(sent, x["x"].numel())]


def _bytes(fmt, n, k):
    return n * k // FORMATS[fmt][1] * FORMATS[fmt][2]


def work(c):
    kind = c["kind"]
    if kind == "linear":
        return {"bytes": _bytes(c["fmt"], c["n"], c["k"]) + 4 * c["rows"] * (c["n"] + c["k"]),
                "flops": 2 * c["rows"] * c["n"] * c["k"]}
    if kind in ("layer", "decode"):
        shapes, h, f = _layer_shapes(c), c["hidden"], c["ffn"]
        ins, outs = 3 * h + f, 2 * h + 2 * c["kv"] + f + h
        return {"bytes": c.get("layers", 1) * (sum(_bytes(t, n, k) for _, t, n, k in shapes)
                                               + 4 * c["rows"] * (ins + outs)),
                "flops": c.get("layers", 1) * 2 * c["rows"] * sum(n * k for _, _, n, k in shapes)}
    if kind == "moe":
        h, f, pairs = c["hidden"], c["width"], c["tokens"] * c["topk"]
        touched = c["experts"] * (1 - (1 - c["topk"] / c["experts"]) ** c["tokens"])  # expected, routed at random
        return {"bytes": touched * (_bytes(c["fmt"], 2 * f, h) + _bytes(c["down"], h, f))
                + 4 * (c["tokens"] * h + pairs * (2 * f + f + h)), "flops": 2 * pairs * 3 * f * h}
    n = c["rows"] * c["hidden"]
    sent = -(-n // 32) * 34
    return {"bytes": (4 * n + sent) + (sent + 4 * n), "flops": 4 * n}


def tolerance(c):
    """About four times what the outputs were seen off their 64-bit values."""
    if c["kind"] == "wire":
        return {"rel": 1e-6}  # the bytes to the last bit, the decoded values products of two 16-bit numbers
    k_quants = {"q4_k", "q6_k"} & {c["fmt"], c.get("down")}
    if c["kind"] in ("linear", "layer") and k_quants and c["rows"] > 2:
        # int8 and f16 operands of the matrix cores: 7e-3 to 9e-3 seen, 6e-4 to 9e-4 from 33 to 128 rows
        return {"rel": 3e-3 if 32 < c["rows"] <= 128 else 2e-2}
    return {"rel": 5e-6}  # exact integer block sums added up in f32: up to 5e-7 seen at the longest rows


def _q8_k(x):
    """The values of an activation quantized per 256 (BlockQ8K): codes of
    -127 / (the value of largest magnitude), rounded half away from zero."""
    b = x.reshape(-1, 256)
    at = b.abs().argmax(1, keepdim=True)
    largest = b.gather(1, at)
    inv = torch.full_like(largest, -127.0) / largest  # one rounding (a scalar's quotient has two)
    t = inv * b
    q = torch.copysign(torch.floor(t.abs().double() + 0.5), t.double()).clamp(-128, 127)
    return (q * (1.0 / inv).double()).reshape(x.shape)


def _over_127(b):
    m = b.abs().amax(1, keepdim=True)
    return m / torch.full_like(m, 127.0)


def _q8_0(x):
    """The values of an activation quantized per 32 (BlockQ8_0)."""
    b = x.reshape(-1, 32)
    d = _over_127(b)
    t = b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    q = torch.copysign(torch.floor(t.abs().double() + 0.5), t.double()).clamp(-128, 127)
    return (q * d.half().double()).reshape(x.shape)


def _product(w, fmt, n, k, a):
    """a (float64, quantized values) times the weight transposed, in 64 bits."""
    step = max(1, CHUNK // k)
    row = k // FORMATS[fmt][1] * FORMATS[fmt][2]
    out = [a @ _values(fmt, w[i * row:min(n, i + step) * row]).view(-1, k).T.contiguous() for i in range(0, n, step)]
    return out[0] if len(out) == 1 else torch.cat(out, -1)


def exact(c, seed):
    w, x = _inputs(c, seed)
    raw = {m: t[2] for m, t in w.items()}

    def times(m, fmt, n, k, v):
        return _product(raw[m], fmt, n, k, _q8_k(v) if FORMATS[fmt][1] == 256 else _q8_0(v))

    if c["kind"] == "linear":
        return times("w", c["fmt"], c["n"], c["k"], x["x"])
    if c["kind"] in ("layer", "decode"):
        outs = []
        for i in range(c.get("layers", 1)):
            xi, tag = (x[i], str(i)) if c["kind"] == "decode" else (x, "")
            y = {m: times(m + tag, f, n, k, xi[{"o": "o", "gate": "mlp", "up": "mlp", "down": "down"}.get(m, "qkv")])
                 for m, f, n, k in _layer_shapes(c)}
            outs.append([y["q"], y["k"], y["v"], y["o"], y["gate"] * torch.sigmoid(y["gate"]) * y["up"], y["down"]])
        return outs if c["kind"] == "decode" else outs[0]
    if c["kind"] == "moe":
        e, h, f, topk = c["experts"], c["hidden"], c["width"], c["topk"]
        prompt = c["tokens"] > 8
        pair_expert = x["experts"].reshape(-1)
        up = torch.zeros((pair_expert.numel(), 2 * f), dtype=torch.float64, device=DEV)
        down = torch.zeros((pair_expert.numel(), h), dtype=torch.float64, device=DEV)
        for name, fmt, n, k, v, out, per_pair in (("gate_up", c["fmt"], 2 * f, h, x["x"], up, False),
                                                  ("down", c["down"], h, f, x["y"], down, True)):
            # a prompt's products take the inputs and weights in f16, the others the quantized inputs
            a = v.half().double() if prompt else _q8_k(v) if FORMATS[fmt][1] == 256 else _q8_0(v)
            row = _bytes(fmt, n, k)
            for ex in range(e):
                pairs = (pair_expert == ex).nonzero().view(-1)
                if not pairs.numel():
                    continue
                vals = _values(fmt, raw[name][ex * row:(ex + 1) * row]).view(n, k)
                vals = vals.float().half().double() if prompt else vals
                got = a[pairs if per_pair else pairs // topk] @ vals.T.contiguous()
                out[pairs] = got * x["topw"][pairs].double()[:, None] if per_pair else got
        return [up, down]
    # the wire bytes are whole values; their decoded form is scale x code
    b = x["x"].reshape(-1, 32)
    d = _over_127(b)
    t = b * (1.0 / d)
    q = torch.copysign(torch.floor(t.abs().double() + 0.5), t.double()).clamp(-127, 127)
    return [None, (q * d.half().double()).reshape(-1)]

"""The work that programs have the quantized-weight path do, as timed cases.

A model's step on this library is linear projections (one activation column
in single-sequence decoding, up to eight in batched decoding), a
512-expert MoE layer (one token when decoding, a few when several sequences
decode together, hundreds to thousands when a prompt is read), the same layer
inside the gated residual, the LM head with its greedy id or with the token
sampler, and whole-tensor dequantization at load time. Shapes are those of
the two layer configurations that the tests and the benchmark run (hidden
2048 with intermediate 512, and hidden 2560 with intermediate 640), their
projections and their LM heads.

Every pass goes through the package's Python binding of the C ABI on one
asynchronous context, as a serving loop does; the sampler returns to the
host by its nature. Weights are random GGUF blocks whose decoded values have
the size of trained weights (about 0.03 rms, zero mean); activations are
N(0, 1), as behind a norm.
"""
from __future__ import annotations

import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT / "kestrel-q_amd"))

import kq_hip  # noqa: E402

DEV = torch.device("cuda", 0)
GEOMETRY = {"Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210), "Q8_0": (32, 34),
            "Q5_1": (32, 24), "IQ4_NL": (32, 18)}
FORMATS = tuple(GEOMETRY)

# hidden, intermediate, the routed gate/up and down formats and the shared
# expert's: the configuration the MoE figures are quoted on, and the two
# kinds of layer of the 2560-wide model. 512 experts, 10 of them per token.
LAYERS = {"2048x512": (2048, 512, "Q4_K", "Q6_K", "Q4_K", "Q6_K"),
          "2560x640": (2560, 640, "Q4_K", "Q5_1", "Q8_0", "Q8_0"),
          "2560x640_q5k": (2560, 640, "Q5_K", "Q8_0", "Q8_0", "Q8_0")}
EXPERTS, TOP_K = 512, 10
BRANCHES, RANK = 4, 320
EPS = 1.0e-6

# LM heads: vocabulary (as stored), columns, format, and the vocabulary's
# ids in use (the sampler refuses ids past them)
HEAD_Q6K = (151936, 2048, "Q6_K")
HEAD_Q8_0 = (248320, 2560, "Q8_0")
CANONICAL = 248077

COLUMNS = (512, 640, 2048, 2560, 4096, 6144, 10240)  # of the projections
MAX_BATCH = 8        # the matvec's own limit
MAX_TOKENS = 2500    # a prompt, or a chunk of one


def listed():
    return [
        # one token's projection, of an odd height: the smallest call, latency and launch
        {"name": "linear_q4_k_4097x2560_b1", "kind": "linear", "fmt": "Q4_K", "rows": 4097,
         "cols": 2560, "batch": 1},
        # eight sequences decoding together through a wide projection
        {"name": "linear_q8_0_10240x2560_b8", "kind": "linear", "fmt": "Q8_0", "rows": 10240,
         "cols": 2560, "batch": 8},
        # the LM head of one sequence, greedy
        {"name": "head_q6_k_151936x2048_b1", "kind": "head", "fmt": "Q6_K", "rows": 151936,
         "cols": 2048, "batch": 1},
        # and of five (an odd number of them), greedy
        {"name": "head_q8_0_248320x2560_b5", "kind": "head", "fmt": "Q8_0", "rows": 248320,
         "cols": 2560, "batch": 5},
        # single-sequence decoding with sampling: LM head and draw in one call
        {"name": "sample_q8_0_248320x2560", "kind": "sample", "top_k": 20, "top_p": 0.95,
         "temperature": 1.0},
        # one token through the MoE layer
        {"name": "moe_2048x512_t1", "kind": "moe", "layer": "2048x512", "tokens": 1},
        # seven sequences decoding together through the Q5_K layer
        {"name": "moe_2560x640_q5k_t7", "kind": "moe", "layer": "2560x640_q5k", "tokens": 7},
        # a prompt of 512 tokens
        {"name": "moe_2048x512_t512", "kind": "moe", "layer": "2048x512", "tokens": 512},
        # a long prompt, of an odd length
        {"name": "moe_2560x640_t2499", "kind": "moe", "layer": "2560x640", "tokens": 2499},
        # the layer inside the gated residual, decoding
        {"name": "block_2560x640_t1", "kind": "block", "layer": "2560x640", "tokens": 1},
        # and on a short prompt
        {"name": "block_2560x640_t201", "kind": "block", "layer": "2560x640", "tokens": 201},
        # a tensor decoded to floats at load time
        {"name": "dequant_q6_k_64m", "kind": "dequant", "fmt": "Q6_K", "blocks": 1 << 18},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(("linear", "linear", "head", "sample", "moe", "moe", "moe", "block",
                       "dequant"))
    if kind == "linear":
        fmt = rng.choice(FORMATS)
        cols = rng.choice([c for c in COLUMNS if c % GEOMETRY[fmt][0] == 0])
        return {"kind": kind, "fmt": fmt, "rows": _log_int(rng, 256, 20000), "cols": cols,
                "batch": rng.randint(1, MAX_BATCH)}
    if kind == "head":
        vocab, cols, fmt = rng.choice((HEAD_Q6K, HEAD_Q8_0))
        return {"kind": kind, "fmt": fmt, "rows": _log_int(rng, 32000, vocab), "cols": cols,
                "batch": rng.randint(1, MAX_BATCH)}
    if kind == "sample":
        return {"kind": kind, "top_k": rng.randint(1, 64), "top_p": round(rng.uniform(0.5, 1.0), 3),
                "temperature": round(rng.uniform(0.5, 1.5), 3)}
    if kind == "dequant":
        fmt = rng.choice(FORMATS)
        per = 256 // GEOMETRY[fmt][0]
        return {"kind": kind, "fmt": fmt, "blocks": _log_int(rng, 1 << 10, 1 << 18) * per + 1}
    layer = rng.choice(tuple(LAYERS) if kind == "moe" else ("2560x640", "2560x640_q5k"))
    return {"kind": kind, "layer": layer,
            "tokens": _log_int(rng, 1, MAX_TOKENS if kind == "moe" else 1000)}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, device=DEV) * (hi - lo) + lo


def _put_half(blocks, at, values):
    blocks[:, at:at + 2] = values.half().view(torch.uint8).reshape(-1, 2)


def _blocks(g, fmt, n):
    """n random GGUF blocks, uint8 [n][bytes]."""
    b = torch.empty((n, GEOMETRY[fmt][1]), dtype=torch.uint8, device=DEV)
    b.view(-1).random_(0, 256, generator=g)
    if fmt in ("Q4_K", "Q5_K"):
        # sub-block scales 16..63, each sub-block's min the same number:
        # dmin takes the codes' mean off
        mid, spread = (7.5, 4.6) if fmt == "Q4_K" else (15.5, 9.2)
        d = _uniform(g, n, 0.5, 1.5) * (0.03 / (41 * spread))
        _put_half(b, 0, d)
        _put_half(b, 2, d * mid)
        sc = torch.randint(16, 64, (n, 8), generator=g, device=DEV, dtype=torch.uint8)
        lo, hi = sc[:, :4], sc[:, 4:]
        b[:, 4:8] = lo | ((hi >> 4) << 6)
        b[:, 8:12] = lo | ((hi >> 4) << 6)
        b[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
    elif fmt == "Q6_K":
        sc = torch.randint(32, 128, (n, 16), generator=g, device=DEV, dtype=torch.int32)
        sign = torch.randint(0, 2, (n, 16), generator=g, device=DEV, dtype=torch.int32) * 2 - 1
        b[:, 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
        _put_half(b, 208, _uniform(g, n, 0.5, 1.5) * (0.03 / (80 * 18.5)))
    elif fmt == "Q8_0":
        _put_half(b, 0, _uniform(g, n, 0.5, 1.5) * (0.03 / 73))
    elif fmt == "Q5_1":
        d = _uniform(g, n, 0.5, 1.5) * (0.03 / 9.2)
        _put_half(b, 0, d)
        _put_half(b, 2, d * -15.5)
    else:
        _put_half(b, 0, _uniform(g, n, 0.5, 1.5) * (0.03 / 66))
    return b


def _matrix(g, fmt, rows, cols):
    be = GEOMETRY[fmt][0]
    return _blocks(g, fmt, rows * (cols // be)).view(rows, -1)


def _normal(g, *shape, sigma=1.0):
    return torch.randn(shape, generator=g, device=DEV) * sigma


def _moe_weights(g, layer):
    h, i, gate, down, sgate, sdown = LAYERS[layer]
    return {"router": _normal(g, EXPERTS, h, sigma=0.02),
            "gate": _matrix(g, gate, EXPERTS * i, h), "up": _matrix(g, gate, EXPERTS * i, h),
            "down": _matrix(g, down, EXPERTS * h, i),
            "shared_gate": _matrix(g, sgate, i, h), "shared_up": _matrix(g, sgate, i, h),
            "shared_down": _matrix(g, sdown, h, i),
            "shared_gate_weight": _normal(g, h, sigma=0.02)}


def _gr_weights(g, h):
    w = BRANCHES * h
    return {"norm": _normal(g, w, sigma=0.1), "down": _matrix(g, "Q8_0", RANK, w),
            "up": _matrix(g, "Q8_0", w, RANK), "inject": _normal(g, BRANCHES, w, sigma=0.01)}


def _inputs(case, seed):
    """The tensors a pass reads; weights first, so that they depend on the
    seed alone and not on the token count."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("linear", "head"):
        return {"w": _matrix(g, case["fmt"], case["rows"], case["cols"]),
                "x": _normal(g, case["batch"], case["cols"])}
    if kind == "sample":
        vocab, cols, fmt = HEAD_Q8_0
        w = _matrix(g, fmt, vocab, cols)
        w.view(vocab, -1, 34)[CANONICAL:, :, :2] = 0  # the padding rows decode to zeros
        return {"w": w, "x": _normal(g, 1, cols)}
    if kind == "dequant":
        return {"w": _blocks(g, case["fmt"], case["blocks"])}
    t, h = case["tokens"], LAYERS[case["layer"]][0]
    t_in = {"moe": _moe_weights(g, case["layer"])}
    if kind == "block":
        t_in["gr"] = _gr_weights(g, h)
        t_in["x"] = _normal(g, t, BRANCHES * h)
    else:
        t_in["x"] = _normal(g, t, h)
    return t_in


# ---------------------------------------------------------------- the passes

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = kq_hip.Context(0)
        _context.set_async(True)
    return _context


class _At:
    """A device tensor under the name that the binding's helpers read."""

    def __init__(self, tensor):
        self.ptr = tensor.data_ptr()


def prepare(case, seed):
    s = {"case": case, "ctx": _ctx(), "in": _inputs(case, seed)}
    kind = case["kind"]
    empty = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device=DEV)  # noqa: E731
    if kind in ("linear", "head"):
        s["y"] = empty(case["batch"], case["rows"])
        s["ids"] = empty(case["batch"], dtype=torch.int32)
    elif kind == "sample":
        s["cfg"] = kq_hip.SamplingConfig(kq_hip.sampling_policy(
            temperature=case["temperature"], top_p=case["top_p"], top_k=case["top_k"]))
        s["rng"] = kq_hip.rng_seed(seed)
        s["y"] = empty(HEAD_Q8_0[0])
        s["scratch"] = empty(s["cfg"].scratch_bytes, dtype=torch.uint8)
    elif kind == "dequant":
        s["y"] = empty(case["blocks"] * GEOMETRY[case["fmt"]][0])
    else:
        h, i, gate, down, sgate, sdown = LAYERS[case["layer"]]
        t, ids = case["tokens"], kq_hip.TYPE_IDS
        s["cfg"] = kq_hip.MoeConfig(h, EXPERTS, TOP_K, i, i)
        s["weights"] = kq_hip.moe_weights({k: _At(v) for k, v in s["in"]["moe"].items()},
                                          ids[gate], ids[down], ids[sgate], ids[sdown])
        s["y"] = torch.empty_like(s["in"]["x"])
        s["ids"] = empty(t, TOP_K, dtype=torch.int32)
        if kind == "block":
            s["dims"] = kq_hip.gr_dims(BRANCHES, h, RANK, EPS)
            s["gr"] = kq_hip.gr_weights({k: _At(v) for k, v in s["in"]["gr"].items()},
                                        kq_hip.TYPE_Q8_0, kq_hip.TYPE_Q8_0)
            n = kq_hip.moe_block_scratch_bytes(s["dims"], s["cfg"], t)
        else:
            n = s["cfg"].scratch_bytes(t)
        s["scratch"] = empty(n, dtype=torch.uint8)
    torch.cuda.synchronize()  # the library's stream is not torch's
    return s


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind == "linear":
        ctx.matvec(kq_hip.TYPE_IDS[case["fmt"]], s["in"]["w"].data_ptr(), case["rows"],
                   case["cols"], s["in"]["x"].data_ptr(), case["batch"], s["y"].data_ptr())
        return s["y"]
    if kind == "head":
        ctx.lm_head(kq_hip.TYPE_IDS[case["fmt"]], s["in"]["w"].data_ptr(), case["rows"],
                    case["cols"], s["in"]["x"].data_ptr(), case["batch"], s["y"].data_ptr(),
                    s["ids"].data_ptr())
        return {"logits": s["y"], "ids": s["ids"]}
    if kind == "sample":
        vocab, cols, fmt = HEAD_Q8_0
        r = ctx.lm_head_sample(s["cfg"], s["rng"], kq_hip.TYPE_IDS[fmt],
                               s["in"]["w"].data_ptr(), vocab, cols, s["in"]["x"].data_ptr(),
                               s["y"].data_ptr(), s["scratch"].data_ptr())
        return {"logits": s["y"], "id": int(r.selected_token_id),
                "retained": int(r.retained_count), "word": int(r.rng_word),
                "probability": float(r.selected_probability),
                "maximum": float(r.maximum_probability)}
    if kind == "dequant":
        w = s["in"]["w"]
        ctx.dequantize(kq_hip.TYPE_IDS[case["fmt"]], w.data_ptr(), w.numel(), s["y"].data_ptr(),
                       s["y"].numel())
        return s["y"]
    x, t = s["in"]["x"].data_ptr(), case["tokens"]
    if kind == "block":
        ctx.moe_block(s["dims"], s["gr"], s["cfg"], s["weights"], x, t, s["y"].data_ptr(),
                      s["ids"].data_ptr(), s["scratch"].data_ptr(), s["scratch"].numel())
    else:
        ctx.moe_execute(s["cfg"], s["weights"], x, t, s["y"].data_ptr(), s["ids"].data_ptr(),
                        s["scratch"].data_ptr(), s["scratch"].numel())
    return {"out": s["y"], "ids": s["ids"]}


# ------------------------------------------------------------ what it costs


def _packed(fmt, rows, cols):
    be, bb = GEOMETRY[fmt]
    return rows * (cols // be) * bb


def work(case):
    kind = case["kind"]
    if kind in ("linear", "head"):
        r, c, b = case["rows"], case["cols"], case["batch"]
        return {"bytes": _packed(case["fmt"], r, c) + 4 * b * (r + c), "flops": 2 * r * c * b}
    if kind == "sample":
        r, c, fmt = HEAD_Q8_0
        return {"bytes": _packed(fmt, r, c) + 4 * (r + c), "flops": 2 * r * c}
    if kind == "dequant":
        be, bb = GEOMETRY[case["fmt"]]
        return {"bytes": case["blocks"] * (bb + 4 * be), "flops": 2 * case["blocks"] * be}
    h, i, gate, down, sgate, sdown = LAYERS[case["layer"]]
    t = case["tokens"]
    # the experts that t tokens of independent choice select
    chosen = EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** t)
    nbytes = (4 * (EXPERTS + 1) * h + chosen * (2 * _packed(gate, i, h) + _packed(down, h, i)) +
              2 * _packed(sgate, i, h) + _packed(sdown, h, i) + 4 * t * TOP_K)
    flops = 2 * t * h * (EXPERTS + 1) + 2 * t * (TOP_K + 1) * 3 * h * i
    width = h
    if kind == "block":
        width = BRANCHES * h
        nbytes += 2 * _packed("Q8_0", RANK, width) + 4 * (BRANCHES + 1) * width
        flops += 2 * t * width * (2 * RANK + BRANCHES)
    return {"bytes": nbytes + 8 * t * width, "flops": flops}


def tolerance(case):
    """About four times the largest error measured against the same sums in
    binary64 (exact): 4.3e-7 of a projection's or a head's binary32 sums over
    512 .. 10240 terms, 1.4e-6 of a MoE layer's three products in a row, and
    3.2e-8 of the block, most of whose output is the residual that it adds
    to. Decoded weights are bits."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind in ("linear", "head", "sample"):
        return {"rel": 2e-6, "max": 2e-5}
    if kind == "block":
        return {"rel": 2e-7, "max": 1e-5}
    return {"rel": 6e-6, "max": 1e-4}


# ---------------------------------------------------------- the same in fp64

_IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _decode(fmt, blocks):
    """Blocks uint8 [n][bytes] to float64 [n][elements]."""
    half = lambda at: blocks[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    n = blocks.shape[0]
    nib = lambda q: (q & 15, q >> 4)  # noqa: E731
    if fmt in ("Q4_K", "Q5_K"):
        q = blocks[:, 4:16]
        lo, mid, hi = q[:, :4], q[:, 4:8], q[:, 8:]
        sc = torch.cat((lo & 63, (hi & 15) | ((lo >> 6) << 4)), 1).double()
        mn = torch.cat((mid & 63, (hi >> 4) | ((mid >> 6) << 4)), 1).double()
        qs = blocks[:, -128:].reshape(n, 4, 32)
        codes = torch.stack(nib(qs), 2).reshape(n, 8, 32)
        if fmt == "Q5_K":
            bit = torch.arange(8, device=blocks.device, dtype=torch.uint8).view(1, 8, 1)
            codes = codes + (((blocks[:, 16:48].reshape(n, 1, 32) >> bit) & 1) << 4)
        w = (half(0) * sc)[:, :, None] * codes.double() - (half(2) * mn)[:, :, None]
        return w.reshape(n, 256)
    if fmt == "Q6_K":
        ql = blocks[:, :128].reshape(n, 2, 2, 32)
        qh = blocks[:, 128:192].reshape(n, 2, 1, 32)
        low = torch.cat(nib(ql), 2)  # [n][half][quarter][32]
        bit = torch.tensor([0, 2, 4, 6], device=blocks.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (low | (((qh >> bit) & 3) << 4)).double() - 32.0
        sc = blocks[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        return (q.reshape(n, 16, 16) * sc[:, :, None]).reshape(n, 256)
    if fmt == "Q8_0":
        return blocks[:, 2:].contiguous().view(torch.int8).double() * half(0)
    codes = torch.cat(nib(blocks[:, -16:]), 1)
    if fmt == "Q5_1":
        bit = torch.arange(8, device=blocks.device, dtype=torch.uint8).view(1, 1, 8)
        fifth = ((blocks[:, 4:8].reshape(n, 4, 1) >> bit) & 1).reshape(n, 32)
        return (codes | (fifth << 4)).double() * half(0) + half(2)
    table = torch.tensor(_IQ4, device=blocks.device, dtype=torch.float64)
    return table[codes.long()] * half(0)


def _linear64(fmt, w, x):
    """x float64 [b][cols] times the packed rows w [rows][bytes], transposed."""
    rows, bb = w.shape[0], GEOMETRY[fmt][1]
    out = torch.empty((x.shape[0], rows), dtype=torch.float64, device=w.device)
    for r in range(0, rows, 16384):
        part = w[r:r + 16384]
        d = _decode(fmt, part.reshape(-1, bb)).reshape(part.shape[0], -1)
        out[:, r:r + 16384] = x @ d.t().contiguous()
    return out


def _expert64(x, gate_fmt, gate, up, down_fmt, down):
    g, u = _linear64(gate_fmt, gate, x), _linear64(gate_fmt, up, x)
    return _linear64(down_fmt, down, g * torch.sigmoid(g) * u)


def _moe64(layer, w, x):
    h, i, gate, down, sgate, sdown = LAYERS[layer]
    logits = x @ w["router"].double().t().contiguous()
    top, ids = torch.topk(logits, TOP_K, dim=1)
    weights = torch.softmax(top, 1)
    out = _expert64(x, sgate, w["shared_gate"], w["shared_up"], sdown, w["shared_down"])
    out *= torch.sigmoid(x @ w["shared_gate_weight"].double())[:, None]
    ids_host = ids.cpu()
    for e in range(EXPERTS):
        tok, slot = (ids_host == e).nonzero(as_tuple=True)
        if not len(tok):
            continue
        tok, slot = tok.to(x.device), slot.to(x.device)
        o = _expert64(x[tok], gate, w["gate"][e * i:(e + 1) * i], w["up"][e * i:(e + 1) * i],
                      down, w["down"][e * h:(e + 1) * h])
        out.index_add_(0, tok, o * weights[tok, slot][:, None])
    return out


def _block64(layer, t_in):
    h, gr = LAYERS[layer][0], t_in["gr"]
    x = t_in["x"].double().view(-1, BRANCHES, h)
    t = x.shape[0]
    inv = (x.square().mean(2, keepdim=True) + EPS).rsqrt()
    norm = (x * inv).reshape(t, -1) * (1.0 + gr["norm"].double())
    r = _linear64("Q8_0", gr["down"], norm) / BRANCHES
    read = torch.sigmoid(_linear64("Q8_0", gr["up"], r * torch.sigmoid(r)))
    mixed = (read * norm).view(t, BRANCHES, h).sum(1) / BRANCHES
    gate = 2.0 * torch.sigmoid(norm @ gr["inject"].double().t().contiguous() / BRANCHES)
    o = _moe64(layer, t_in["moe"], mixed)
    return (x + gate[:, :, None] * o[:, None, :]).reshape(t, -1)


def exact(case, seed):
    t_in, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return _linear64(case["fmt"], t_in["w"], t_in["x"].double())
    if kind == "head":
        return {"logits": _linear64(case["fmt"], t_in["w"], t_in["x"].double()), "ids": None}
    if kind == "sample":
        y = _linear64(HEAD_Q8_0[2], t_in["w"], t_in["x"].double())[0]
        return {"logits": y, "id": None, "retained": None, "word": None, "probability": None,
                "maximum": None}
    if kind == "dequant":
        return _decode(case["fmt"], t_in["w"]).reshape(-1)
    if kind == "block":
        return {"out": _block64(case["layer"], t_in), "ids": None}
    return {"out": _moe64(case["layer"], t_in["moe"], t_in["x"].double()), "ids": None}

"""What the library is used for, as timed cases: one MoE layer (or a short stack of them) on decode tokens, verify
windows and prefill chunks, at the geometries of bench.py and tests/ and at generic ones, plus the pieces a program
calls by themselves (one EXL3 linear, the router logits).

A case is a dict of plain values:
  kind    "moe"     gfr_moe.Moe.run: router logits -> gate -> grouping -> EXL3 experts (the shared one EXL3) -> combine
          "fp8"     gfr_moe.Moe.run_fp8: the same with GLM's gate and the FP8 shared expert of the layer
          "linear"  gfr_moe.Linear.run: one fp16 token through one EXL3 matrix
          "router"  gfr_moe.router_logits: the router's product of a window's hidden rows
  hidden, inter, routed, topk, bits, rows, layers   the layer's shape (bits "2345": layer l has 2 + l bits)
  skew    the Zipf exponent of the experts' popularity (0: uniform)

Several layers a pass stand for the layers a token goes through one after the other: each has weights, a hidden row
and an engine of its own, so that a decode pass finds its weights in HBM and not in a cache, as in a whole model.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "glm-flash-rs_amd"))
import gfr_moe  # noqa: E402

# (hidden, inter, routed, topk) of the benchmark's layers, and the EXL3 + FP8 layer of the served model's geometry
SMALL = dict(hidden=2048, inter=1536, routed=64, topk=4)
WIDE = dict(hidden=5120, inter=1536, routed=160, topk=8)
FP8 = dict(hidden=4096, inter=512, routed=288, topk=8)
LIMIT = 10.0          # the limited SwiGLU's bound
GLM_SCALE = 2.5       # GLM's gate: the routed weights' scale


def listed():
    return [
        # the smallest call: one token through one quantized projection
        dict(name="linear 1 row", kind="linear", hidden=2048, inter=1536, bits=4),
        # single-stream generation: one token through the layers of a model
        dict(name="decode 1 row", kind="moe", rows=1, layers=8, bits="4", skew=0.0, **SMALL),
        # the same at a wider model, its layers quantized to different widths
        dict(name="decode 1 row wide 2345", kind="moe", rows=1, layers=4, bits="2345", skew=1.1, **WIDE),
        # the same with the served model's layer: 288 small experts, GLM's gate, the FP8 shared expert
        dict(name="decode 1 row fp8", kind="fp8", rows=1, layers=4, bits="4", skew=1.1, **FP8),
        # a short speculative window, or a few streams at once
        dict(name="decode 3 rows", kind="moe", rows=3, layers=4, bits="4", skew=1.1, **SMALL),
        # a verify window of the served model (at most 16 rows)
        dict(name="verify 12 rows fp8", kind="fp8", rows=12, layers=2, bits="4", skew=1.1, **FP8),
        # a verify window of several streams (4 streams x 8 drafts)
        dict(name="verify 32 rows", kind="moe", rows=32, layers=1, bits="4", skew=1.1, **SMALL),
        # the tail of a prompt: an odd number of rows, three bits
        dict(name="chunk 77 rows wide", kind="moe", rows=77, layers=1, bits="3", skew=1.1, **WIDE),
        # a short prompt at the widest format
        dict(name="prefill 709 rows wide", kind="moe", rows=709, layers=1, bits="5", skew=1.1, **WIDE),
        # the largest: a full prefill chunk
        dict(name="prefill 8192 rows", kind="moe", rows=8192, layers=1, bits="4", skew=0.0, **SMALL),
        # a full prefill window of the served model, its shared expert on the prepared bf16 weights
        dict(name="prefill 4096 rows fp8", kind="fp8", rows=4096, layers=1, bits="4", skew=1.1, **FP8),
        # the router's product for that window
        dict(name="router 4096 rows", kind="router", rows=4096, hidden=4096, routed=288),
    ]


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe", "fp8", "fp8", "linear", "router"])

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "linear":
        return dict(kind=kind, hidden=256 * spread(4, 32), inter=256 * spread(2, 32), bits=rng.randint(2, 5))
    if kind == "router":
        return dict(kind=kind, rows=spread(1, 4096), hidden=8 * spread(128, 640), routed=rng.randint(32, 288))
    if kind == "fp8":
        shape = FP8 if rng.random() < 0.5 else dict(hidden=512 * rng.randint(2, 10), inter=256 * rng.randint(1, 6),
                                                    routed=rng.randint(32, 288), topk=rng.randint(2, 8))
    else:
        shape = rng.choice([SMALL, WIDE, dict(hidden=256 * rng.randint(4, 20), inter=256 * rng.randint(1, 8),
                                              routed=rng.randint(16, 192), topk=rng.randint(1, 8))])
    # at most the work of the largest listed case, and a state of a few GB
    per_row = (shape["topk"] + 1) * 3 * shape["hidden"] * shape["inter"]
    most = max(1, min(8192 if kind == "moe" else 4096, 8192 * 5 * 3 * 2048 * 1536 // per_row))
    rows = spread(1, most)
    bits = str(rng.randint(2, 5))
    layers = 4 if rows <= 4 else 1
    return dict(kind=kind, rows=rows, layers=layers, bits=bits, skew=rng.choice([0.0, 0.6, 1.1]), **shape)


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _words(g, *shape):
    return torch.randint(-(2 ** 31), 2 ** 31, shape, generator=g, dtype=torch.int32, device="cuda")


def _scale(g, size, *shape):
    """Column scales: random signs, magnitudes spread around `size`."""
    sign = torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.int32) * 2 - 1
    return (sign * (torch.rand(shape, generator=g, device="cuda") + 0.5) * size).to(torch.float16)


def _experts(g, E, hidden, inter, bits):
    """Random trellis words (every bit string is a valid tensor). The output scales make a layer's values of order one,
    as a quantized model's do, so that the SwiGLU's limit is met now and then and not everywhere. (A codebook value's
    standard deviation is about 1.24.)"""
    D, N, W = hidden, inter, 8 * bits
    return gfr_moe.Exl3Experts(
        gt=_words(g, E, D // 16, N // 16, W), ut=_words(g, E, D // 16, N // 16, W),
        dt=_words(g, E, N // 16, D // 16, W),
        suh_g=_scale(g, 1.0, E, D), suh_u=_scale(g, 1.0, E, D), suh_d=_scale(g, 1.0, E, N),
        svh_g=_scale(g, 2.0 / (1.24 * D ** 0.5), E, N), svh_u=_scale(g, 2.0 / (1.24 * D ** 0.5), E, N),
        svh_d=_scale(g, 1.0 / (1.24 * N ** 0.5), E, D), bits=bits)


def _fp8_shared(g, hidden, inter):
    def mat(n, k):
        return (torch.randn((n, k), generator=g, device="cuda") * 16).to(torch.float8_e4m3fn)

    def sc(n, k, size):
        return ((torch.rand(n, generator=g, device="cuda") + 0.5) * size / (16 * k ** 0.5)).to(torch.bfloat16)

    return gfr_moe.Fp8SharedWeights(gu=mat(2 * inter, hidden), gu_scale=sc(2 * inter, hidden, 2.0),
                                    down=mat(hidden, inter), down_scale=sc(hidden, inter, 1.0))


def _logits(g, rows, routed, skew):
    """Router logits whose picks follow a Zipf popularity of the experts (skew 0: uniform)."""
    u = torch.rand((rows, routed), generator=g, device="cuda").clamp_(1e-7, 1 - 1e-7)
    gumbel = -torch.log(-torch.log(u))
    rank = torch.randperm(routed, generator=g, device="cuda").float() + 1
    return (gumbel - skew * torch.log(rank)).contiguous()


def _rows(g, rows, hidden):
    return torch.randn((rows, hidden), generator=g, device="cuda").to(torch.bfloat16)


def _bits(case, layer):
    return int(case["bits"]) if len(case["bits"]) == 1 else int(case["bits"][layer])


def _layer_inputs(case, seed, layer):
    """One layer's weights and inputs, from the seed alone."""
    g = _gen(seed * 64 + layer)
    fp8 = case["kind"] == "fp8"
    E = case["routed"] + (0 if fp8 else 1)
    d = dict(w=_experts(g, E, case["hidden"], case["inter"], _bits(case, layer)),
             x=_rows(g, case["rows"], case["hidden"]),
             logits=_logits(g, case["rows"], case["routed"], case["skew"]))
    if fp8:
        d["logits"] *= 0.5                       # sigmoid scores away from saturation
        d["shared"] = _fp8_shared(g, case["hidden"], case["inter"])
        d["bias"] = torch.randn(case["routed"], generator=g, device="cuda") * 0.02
    return d


def _linear_inputs(case, seed):
    g = _gen(seed * 64)
    k, n = case["hidden"], case["inter"]
    return dict(x=torch.randn(k, generator=g, device="cuda").half(), t=_words(g, k // 16, n // 16, 8 * case["bits"]),
                suh=_scale(g, 1.0, k), svh=_scale(g, 1.0 / (1.24 * k ** 0.5), n))


def _router_inputs(case, seed):
    g = _gen(seed * 64)
    w = (torch.randn((case["routed"], case["hidden"]), generator=g, device="cuda") / case["hidden"] ** 0.5)
    return dict(x=_rows(g, case["rows"], case["hidden"]), w=w.to(torch.bfloat16))


class Outputs(list):
    """A pass's outputs: views of the engines' own buffers, valid while the engines live, so it holds the engines."""


def prepare(case, seed):
    if case["kind"] == "linear":
        s = _linear_inputs(case, seed)
        s["engine"] = gfr_moe.Linear(case["hidden"], case["inter"], case["bits"])
        s["y"] = torch.empty(case["inter"], dtype=torch.float32, device="cuda")
    elif case["kind"] == "router":
        s = _router_inputs(case, seed)
    else:
        fp8 = case["kind"] == "fp8"
        s = dict(layers=[], out=Outputs())
        s["out"].engines = []
        for layer in range(case["layers"]):
            d = _layer_inputs(case, seed, layer)
            d["moe"] = gfr_moe.Moe(case["hidden"], case["inter"], case["routed"], case["topk"], case["rows"],
                                   shared_exl3=not fp8)
            if fp8:
                d["moe"].set_router(d["bias"], GLM_SCALE)
                d["shared"].prepare_bf16()       # a program that also prefills holds the bf16 copies
            s["layers"].append(d)
            s["out"].append({"out": d["moe"].output, "picks": d["moe"].picks, "weights": d["moe"].weights})
            s["out"].engines.append(d["moe"])
    return dict(s, kind=case["kind"], rows=case.get("rows", 1))


def run(state):
    kind, rows = state["kind"], state["rows"]
    if kind == "linear":
        state["engine"].run(state["x"], state["t"], state["suh"], state["svh"], state["y"])
        return state["y"]
    if kind == "router":
        return gfr_moe.router_logits(state["x"], state["w"])
    for d in state["layers"]:
        if kind == "fp8":
            d["moe"].run_fp8(d["w"], d["x"], d["logits"], d["shared"], rows)
        else:
            d["moe"].run(d["w"], d["x"], d["logits"], rows)
    return state["out"]


# ---- the work of a pass -----------------------------------------------------------------------------------------------
def _distinct(case):
    """Expected distinct routed experts of a window: each row draws topk of them without replacement by popularity."""
    E, k, rows = case["routed"], case["topk"], case["rows"]
    p = [1.0 / (r + 1) ** case["skew"] for r in range(E)]
    total = sum(p)
    p = [v / total for v in p]
    # the rate c at which a row's picks cover expert e with probability 1 - exp(-c p_e), sum over e = topk
    lo, hi = 0.0, 1e9
    for _ in range(80):
        c = (lo + hi) / 2
        if sum(1 - math.exp(-c * v) for v in p) < min(k, E - 1e-6):
            lo = c
        else:
            hi = c
    return sum(1 - math.exp(-rows * c * v) for v in p)


def work(case):
    if case["kind"] == "linear":
        k, n = case["hidden"], case["inter"]
        return {"bytes": k * n * case["bits"] / 8 + 2 * k + 2 * k + 2 * n + 4 * n, "flops": 2 * k * n}
    if case["kind"] == "router":
        m, k, n = case["rows"], case["hidden"], case["routed"]
        return {"bytes": 2 * m * k + 2 * n * k + 4 * m * n, "flops": 2 * m * n * k}
    D, N, rows, k = case["hidden"], case["inter"], case["rows"], case["topk"]
    total = {"bytes": 0.0, "flops": 0.0}
    for layer in range(case["layers"]):
        one = 3 * D * N * _bits(case, layer) / 8 + 2 * (3 * D + 3 * N)
        # the shared expert: one more EXL3 expert, or the FP8 one
        shared = one if case["kind"] == "moe" else 3 * D * N + 2 * (2 * N + D)
        io = rows * (2 * D + 4 * D + 4 * case["routed"] + 8 * (k + 1))
        total["bytes"] += _distinct(case) * one + shared + io
        total["flops"] += rows * (k + 1) * 2 * 3 * D * N
    return total


def tolerance(case):
    # picks are whole numbers and stay the same; weights are 32-bit sums over the picks
    if case["kind"] == "router":
        return {"rel": 1e-5, "max": 1e-4}        # 32-bit sums in another order
    if case["kind"] == "linear":
        return {"rel": 1.5e-3, "max": 1.5e-2}    # the weight as an fp16 value or as the sum of its two halves
    # fp16 rows, the SwiGLU's bf16 roundings: one rounding the other way here and there
    return {"rel": 6e-3, "max": 1e-1}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------
def _codebook():
    """The value of each 16-bit state: x = s * 0xCBAC1FED mod 2^32, (x & 0x8FFF8FFF) ^ 0x3B603B60 read as two fp16
    halves, their sum rounded to fp16."""
    s = torch.arange(65536, dtype=torch.int64, device="cuda")
    x = (s * 0xCBAC1FED) & 0xFFFFFFFF
    x = (x & 0x8FFF8FFF) ^ 0x3B603B60

    def half(v):
        return (v & 0xFFFF).to(torch.int32).to(torch.int16).view(torch.float16)

    return (half(x).double() + half(x >> 16).double()).to(torch.float16).double()


def _decode(words, table):
    """[KT, NT, 8 K] trellis words -> [16 KT, 16 NT] weights in 64 bits: value p of a tile is the 16-bit window of the
    circular bit stream that ends at bit (p + 1) K, at row 2 (L % 4) + (j & 1) + 8 ((j >> 1) & 1) and column
    L / 4 + 8 (j >> 2), L = p / 8, j = p % 8."""
    KT, NT, W = words.shape
    bits = W // 8
    p = torch.arange(256, device="cuda")
    start = ((p + 1) * bits - 16) % (32 * W)
    first, off = start // 32, start % 32
    L, j = p // 8, p % 8
    row, col = 2 * (L % 4) + (j & 1) + 8 * ((j >> 1) & 1), L // 4 + 8 * (j >> 2)
    out = torch.empty((KT, 16, NT, 16), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 24) // (NT * 256))
    for k0 in range(0, KT, step):
        w = words[k0:k0 + step].to(torch.int64) & 0xFFFFFFFF
        pair = (w[..., first] << 32) | w[..., (first + 1) % W]
        state = (pair >> (48 - off)) & 0xFFFF
        part = torch.empty((w.shape[0], 16, NT, 16), dtype=torch.float64, device="cuda")
        part[:, row, :, col] = table[state].permute(2, 0, 1)
        out[k0:k0 + step] = part
    return out.view(KT * 16, NT * 16)


def _had(x):
    """The orthonormal 128-point Walsh-Hadamard transform of each block of 128 along the last dimension."""
    h = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    while h.shape[0] < 128:
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return ((x.view(-1, 128) @ h) / math.sqrt(128)).view(x.shape)


def _swiglu(g, u):
    g = g.clamp(max=LIMIT)
    return g / (1 + torch.exp(-g)) * u.clamp(-LIMIT, LIMIT)


def _expert(d, e, x, table):
    w = d["w"]

    def v(name):
        return getattr(w, name)[e].double()

    g = _had(_had(x * v("suh_g")) @ _decode(w.gt[e], table)) * v("svh_g")
    u = _had(_had(x * v("suh_u")) @ _decode(w.ut[e], table)) * v("svh_u")
    a = _had(_swiglu(g, u) * v("suh_d"))
    return _had(a @ _decode(w.dt[e], table)) * v("svh_d")


def _exact_layer(case, seed, layer, table):
    d = _layer_inputs(case, seed, layer)
    rows, k = case["rows"], case["topk"]
    x, logits = d["x"].double(), d["logits"].double()
    out = torch.zeros((rows, case["hidden"]), dtype=torch.float64, device="cuda")
    if case["kind"] == "fp8":
        score = torch.sigmoid(logits)
        picks = torch.topk(score + d["bias"].double(), k, dim=1).indices
        weights = score.gather(1, picks)
        weights = weights / (weights.sum(1, keepdim=True) + 1e-20) * GLM_SCALE
        sw = d["shared"]
        gu = (x @ sw.gu.double().t()) * sw.gu_scale.double()
        act = _swiglu(gu[:, :case["inter"]], gu[:, case["inter"]:])
        out += (act @ sw.down.double().t()) * sw.down_scale.double()
    else:
        top, picks = torch.topk(logits, k, dim=1)
        weights = torch.softmax(top, dim=1)
        out += _expert(d, case["routed"], x, table)
    for e in picks.unique().tolist():
        r, s = (picks == e).nonzero(as_tuple=True)
        out[r] += weights[r, s].unsqueeze(1) * _expert(d, e, x[r], table)
    one = torch.ones((rows, 1), dtype=torch.float64, device="cuda")
    return {"out": out, "picks": None, "weights": torch.cat((weights, one), 1)}


def exact(case, seed):
    if case["kind"] == "router":
        s = _router_inputs(case, seed)
        return s["x"].double() @ s["w"].double().t()
    table = _codebook()
    if case["kind"] == "linear":
        s = _linear_inputs(case, seed)
        x = _had(s["x"].double() * s["suh"].double())
        return _had((x.view(1, -1) @ _decode(s["t"], table)).view(-1)) * s["svh"].double()
    return [_exact_layer(case, seed, layer, table) for layer in range(case["layers"])]

"""The int8 path's work as a user's program has it done, case by case.

Every case goes through mlfw_amd.ops or mlfw_amd.configs.  Small calls are
made the way a serving loop makes them: whole sequences captured once in a
HIP graph and replayed, single calls validated once with ops.prepare.

Kinds and the ranges their drawn cases take:

  mlp      a quantized MLP classifier, 784 -> h1 -> h2 -> 10, batch 1..1024
           (the framework's C2 workload: per-tensor dynamic activations)
  decode   the four linears of a decoder layer and its gated activation for
           1..16 tokens, hidden 1024..5120, feed-forward 2.5..4 times that
  linear   one dynamic per-token linear, 17..4096 tokens, any K and N from
           256 to 12288, with and without bias and activation
  prefill  the decoder projection set (the C4 workload), 64..2048 tokens
  quant    per-token quantize of an activation tensor with outliers, and
           the dequantize of its codes, up to 2^26 elements
  conv     quantized_conv of a batch of images, symmetric int8 or affine
           (ui8 activations with a zero point), fp32 out
  w4       a gated MLP block with 4-bit per-group weights, 1..512 tokens
  dot      quantized_dot of the affine scheme (zero points, ui8 operands),
           int32 out, any sizes

Every result of this path is fixed to the bit (int8 codes, int32 sums and
fp32 outputs follow one rounding sequence, and integer sums do not depend on
their order), so every case compares exactly.
"""
import math

import torch
import torch.nn.functional as F

from mlfw_amd import configs, ops

DEV = "cuda:0"


def listed():
    return [
        # the smallest call: a classifier's forward on one batch of a test or tool
        {"name": "mlp_b256", "kind": "mlp", "batch": 256, "h1": 256, "h2": 128},
        # one sequence decoding: latency per layer, every weight read once
        {"name": "decode_1", "kind": "decode", "tokens": 1, "hidden": 4096, "ff": 11008},
        # sixteen sequences decoding together
        {"name": "decode_16", "kind": "decode", "tokens": 16, "hidden": 4096, "ff": 11008},
        # a larger decode batch or a short prompt through one projection
        {"name": "linear_64", "kind": "linear", "M": 64, "N": 11008, "K": 4096, "bias": False, "act": "none"},
        # the large square product the benchmark's headline is quoted on
        {"name": "linear_4096", "kind": "linear", "M": 4096, "N": 4096, "K": 4096, "bias": False, "act": "none"},
        # a prompt of 2048 tokens through a whole layer's projections
        {"name": "prefill_2048", "kind": "prefill", "tokens": 2048},
        # activation tensors quantized and read back between fp32 layers
        {"name": "quant_16384", "kind": "quant", "M": 16384, "K": 4096},
        # a ResNet stage's 3 x 3 layer on a batch of 32, symmetric scheme, weight prepacked once
        {"name": "conv_56", "kind": "conv", "n": 32, "c": 64, "h": 56, "w": 56, "o": 64, "k": 3, "stride": 1,
         "pad": 1, "groups": 1, "u8": False, "zp": 0},
        # the next stage's layer in the affine scheme: ui8 activations with a zero point
        {"name": "conv_affine", "kind": "conv", "n": 32, "c": 128, "h": 28, "w": 28, "o": 128, "k": 3, "stride": 1,
         "pad": 1, "groups": 1, "u8": True, "zp": 117},
        # 4-bit weights: a few sequences decoding, and a prompt
        {"name": "w4_4", "kind": "w4", "tokens": 4, "hidden": 4096, "ff": 11008, "group": 128},
        {"name": "w4_256", "kind": "w4", "tokens": 256, "hidden": 4096, "ff": 11008, "group": 128},
        # an affine linear (ui8 activations) at sizes that no tile divides
        {"name": "dot_affine", "kind": "dot", "M": 788, "N": 1000, "K": 1500, "u8": True, "zpA": 121, "zpB": 0},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mult(v, m):
    return max(m, v // m * m)


def draw(rng):
    kind = rng.choice(["mlp", "decode", "linear", "linear", "prefill", "quant", "conv", "conv", "w4", "dot"])
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 1, 1024), "h1": _log(rng, 32, 1024), "h2": _log(rng, 16, 512)}
    if kind == "decode":
        hidden = _mult(rng.randint(1024, 5120), 64)
        return {"kind": kind, "tokens": rng.randint(1, 16), "hidden": hidden,
                "ff": _mult(int(hidden * rng.uniform(2.5, 4.0)), 32)}
    if kind == "linear":
        while True:
            M, N, K = _log(rng, 17, 4096), _log(rng, 256, 12288), _log(rng, 256, 12288)
            if rng.random() < 0.75:      # most layers' widths are multiples of 16, some are not
                K = _mult(K, rng.choice([16, 64, 128]))
            if M * N * K <= 4096 ** 3 and (K % 16 == 0 or M * N * K <= 1 << 32):
                break
        return {"kind": kind, "M": M, "N": N, "K": K, "bias": rng.random() < 0.5,
                "act": rng.choice(["none", "none", "relu", "silu"])}
    if kind == "prefill":
        return {"kind": kind, "tokens": _log(rng, 64, 2048)}
    if kind == "quant":
        while True:
            M, K = _log(rng, 16, 16384), _log(rng, 64, 16384)
            if 1 << 14 <= M * K <= 1 << 26:
                return {"kind": kind, "M": M, "K": K}
    if kind == "conv":
        while True:
            u8 = rng.random() < 0.4
            groups = rng.choice([1, 1, 1, 1, 2, 4])
            c = groups * rng.choice([3, 16, 24, 32, 48, 64, 96, 128, 256, 512])
            o = groups * rng.choice([16, 24, 32, 48, 64, 96, 128, 256, 512])
            h = rng.choice([7, 13, 14, 17, 28, 35, 56, 112])
            k = rng.choice([1, 3, 3, 3, 5, 7])
            case = {"kind": kind, "n": _log(rng, 1, 32), "c": c, "h": h, "w": h + rng.choice([0, 0, 0, 3]), "o": o,
                    "k": k, "stride": rng.choice([1, 1, 2]), "pad": k // 2, "groups": groups, "u8": u8,
                    "zp": rng.randint(0, 255) if u8 else 0}
            if 1 << 22 <= work(case)["flops"] <= 7.4e9:
                return case
    if kind == "w4":
        group = rng.choice([32, 64, 128, 128])
        hidden = _mult(rng.randint(1024, 4096), 128)
        return {"kind": kind, "tokens": _log(rng, 1, 512), "hidden": hidden,
                "ff": _mult(int(hidden * rng.uniform(2.0, 3.0)), 128), "group": group}
    while True:
        u8 = rng.random() < 0.5
        M, N, K = _log(rng, 17, 2048), _log(rng, 16, 4096), _log(rng, 64, 4096)
        if M * N * K <= 1 << 32:
            return {"kind": "dot", "M": M, "N": N, "K": K, "u8": u8,
                    "zpA": rng.randint(0, 255) if u8 else rng.randint(-128, 127),
                    "zpB": 0 if rng.random() < 0.7 else rng.randint(-20, 20)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, shape, std=1.0):
    return torch.randn(shape, device=DEV, generator=g) * std


def _inputs(case, seed):
    """Everything the seed decides: activations N(0, 1), weights N(0, 0.02) or
    N(0, 1 / fan_in), codes over the whole range of their type."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "mlp":
        dims = (784, case["h1"], case["h2"], 10)
        return {"x": torch.rand((case["batch"], 784), device=DEV, generator=g),
                "W": [_normal(g, (dims[i + 1], dims[i]), dims[i] ** -0.5) for i in range(3)]}
    if kind == "decode":
        T, H, f = case["tokens"], case["hidden"], case["ff"]
        return {"x": _normal(g, (T, H)), "attn": _normal(g, (T, H)),
                "W": {"qkv": _normal(g, (3 * H, H), 0.02), "o": _normal(g, (H, H), 0.02),
                      "gate_up": _normal(g, (2 * f, H), 0.02), "down": _normal(g, (H, f), 0.02)}}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"x": _normal(g, (M, K)), "W": _normal(g, (N, K), 0.02),
                "bias": torch.rand(N, device=DEV, generator=g) * 0.2 - 0.1 if case["bias"] else None}
    if kind == "prefill":
        return {"X": _normal(g, (case["tokens"], 4096)),
                "W": {k: _normal(g, s, 0.02) for k, s in configs.C4_SHAPES.items()}}
    if kind == "quant":
        x = _normal(g, (case["M"], case["K"]))
        x[torch.rand(x.shape, device=DEV, generator=g) < 0.01] *= 50.0
        return {"x": x}
    if kind == "conv":
        lo, hi, dt = (0, 256, torch.uint8) if case["u8"] else (-128, 128, torch.int8)
        x = torch.randint(lo, hi, (case["n"], case["c"], case["h"], case["w"]), device=DEV, generator=g, dtype=dt)
        w = torch.randint(-127, 128, (case["o"], case["c"] // case["groups"], case["k"], case["k"]), device=DEV,
                          generator=g, dtype=torch.int8)
        return {"x": x, "w": w, "s_out": 1.3e-4}
    if kind == "w4":
        T, H, f = case["tokens"], case["hidden"], case["ff"]
        return {"x": _normal(g, (T, H)), "W": {"gate_up": _normal(g, (2 * f, H), 0.02), "down": _normal(g, (H, f), 0.02)}}
    lo, hi, dt = (0, 256, torch.uint8) if case["u8"] else (-128, 128, torch.int8)
    return {"A": torch.randint(lo, hi, (case["M"], case["K"]), device=DEV, generator=g, dtype=dt),
            "B": torch.randint(-127, 128, (case["N"], case["K"]), device=DEV, generator=g, dtype=torch.int8)}


# ------------------------------------------------------------------ the calls
def _captured(fn):
    """fn's launches in one HIP graph, and what fn returned inside it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _decode(x, attn, P):
    qkv, _, _ = ops.qlinear_dynamic(x, *P["qkv"])
    o, _, _ = ops.qlinear_dynamic(attn, *P["o"])
    gu, _, _ = ops.qlinear_dynamic(o, *P["gate_up"])
    f = gu.shape[1] // 2
    hq, sh = ops.silu_mul_quantize(gu[:, :f], gu[:, f:])
    return {"qkv": qkv, "o": o, "gate_up": gu, "hq": hq, "sh": sh, "down": ops.qlinear(hq, sh, *P["down"])}


def _w4_block(x, P, hidden, ff, group):
    xq, sx = ops.quantize_per_token(x)
    gu = ops.qlinear_w4(xq, sx, *P["gate_up"], hidden, group)
    hq, sh = ops.silu_mul_quantize(gu[:, :ff], gu[:, ff:])
    return {"xq": xq, "sx": sx, "gate_up": gu, "hq": hq, "sh": sh,
            "down": ops.qlinear_w4(hq, sh, *P["down"], ff, group)}


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        packed = configs.c2_prepare(inp["W"])
        graph, out = _captured(lambda: configs.c2_run(inp["x"], packed))
        return {"replay": graph, "out": out, "keep": (inp["x"], packed)}
    if kind == "decode":
        P = {k: ops.pack_weight(w) for k, w in inp["W"].items()}
        graph, out = _captured(lambda: _decode(inp["x"], inp["attn"], P))
        return {"replay": graph, "out": out, "keep": (inp["x"], inp["attn"], P)}
    if kind == "linear":
        W = ops.pack_weight(inp["W"])
        call = ops.prepare(ops.qlinear_dynamic, inp["x"], *W, bias=inp["bias"], act=case["act"])
        return {"calls": [call], "out": call.outputs, "keep": (inp["x"], W, inp["bias"])}
    if kind == "prefill":
        return {"step": (inp["X"], configs.c4_prepare(inp["W"]))}
    if kind == "quant":
        q = ops.prepare(ops.quantize_per_token, inp["x"])
        d = ops.prepare(ops.dequantize, *q.outputs)
        return {"calls": [q, d], "out": (*q.outputs, d.outputs), "keep": inp["x"]}
    if kind == "conv":
        x, w, s, p = inp["x"], inp["w"], [case["stride"]] * 2, [[case["pad"]] * 2] * 2
        taps = None if case["u8"] else ops.conv_weight_taps(w, case["groups"])
        call = ops.prepare(ops.quantized_conv, x, w, s, p, groups=case["groups"], s_out=inp["s_out"], zpx=case["zp"],
                           w_taps=taps)
        return {"calls": [call], "out": call.outputs, "keep": (x, w, taps)}
    if kind == "w4":
        P = {k: ops.pack_weight_int4(w, case["group"]) for k, w in inp["W"].items()}
        graph, out = _captured(lambda: _w4_block(inp["x"], P, case["hidden"], case["ff"], case["group"]))
        return {"replay": graph, "out": out, "keep": (inp["x"], P)}
    return {"dot": (inp["A"], inp["B"], case["zpA"], case["zpB"])}


def run(state):
    if "replay" in state:
        state["replay"].replay()
        return state["out"]
    if "calls" in state:
        for call in state["calls"]:
            call()
        return state["out"]
    if "step" in state:
        return configs.c4_step(*state["step"])
    return ops.quantized_dot(*state["dot"])


# ------------------------------------------------------------------ bounds
def work(case):
    """Bytes: every input and weight of the call read once, every output it
    returns written once; flops: two per multiply-accumulate."""
    kind = case["kind"]
    if kind == "mlp":
        b, d = case["batch"], (784, case["h1"], case["h2"], 10)
        macs = sum(d[i] * d[i + 1] for i in range(3))
        return {"bytes": 4 * b * 784 + macs + 8 * sum(d[1:]) + 40 * b, "flops": 2 * b * macs}
    if kind in ("decode", "w4"):
        T, H, f = case["tokens"], case["hidden"], case["ff"]
        if kind == "decode":
            w = 3 * H * H + H * H + 3 * f * H
            scales, io = 8 * (5 * H + 2 * f), 8 * T * H + 4 * T * (3 * H + H + 2 * f + H) + T * (f + 8)
            return {"bytes": w + scales + io, "flops": 2 * T * w}
        w = 3 * f * H
        return {"bytes": w // 2 + 8 * w // case["group"] + 4 * T * H + T * (H + 8) + 4 * T * (2 * f + H) + T * (f + 8),
                "flops": 2 * T * w}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * M * K + M * K + 8 * M + N * K + 8 * N + 4 * M * N + (4 * N if case["bias"] else 0),
                "flops": 2 * M * N * K}
    if kind == "prefill":
        T = case["tokens"]
        w = sum(n * k for n, k in configs.C4_SHAPES.values())
        outs = 4 * T * (12288 + 4096 + 22016 + 4096) + T * (3 * 4096 + 11008) + 8 * T * 4
        return {"bytes": 4 * T * 4096 + w + 8 * (12288 + 4096 + 22016 + 4096) + outs, "flops": 2 * T * w}
    if kind == "quant":
        n = case["M"] * case["K"]
        return {"bytes": 4 * n + n + 8 * case["M"] + 4 * n, "flops": 2 * n}
    if kind == "conv":
        cg = case["c"] // case["groups"]
        ho = (case["h"] + 2 * case["pad"] - case["k"]) // case["stride"] + 1
        wo = (case["w"] + 2 * case["pad"] - case["k"]) // case["stride"] + 1
        kc, outs = cg * case["k"] ** 2, case["n"] * case["o"] * ho * wo
        return {"bytes": case["n"] * case["c"] * case["h"] * case["w"] + case["o"] * kc + 4 * outs, "flops": 2 * outs * kc}
    M, N, K = case["M"], case["N"], case["K"]
    return {"bytes": M * K + N * K + 4 * M * N, "flops": 2 * M * N * K}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------ in 64 bits
def _q64(x, tensor=False):
    """Symmetric dynamic codes and scale of x in 64 bits."""
    x = x.double()
    s = x.abs().max() / 127 if tensor else x.abs().amax(1, keepdim=True) / 127
    s = torch.where(s == 0, torch.full_like(s, 1e-10), s)
    return torch.clamp(torch.floor(x / s + 0.5), -128, 127), s


def _w64(W, group=None):
    """The weight as its codes say: codes times scales, in 64 bits."""
    W = W.double()
    if group is None:
        s = W.abs().amax(1, keepdim=True) / 127
        return torch.clamp(torch.floor(W / s + 0.5), -128, 127) * s
    G = W.reshape(-1, group)
    s = G.abs().amax(1, keepdim=True) / 7
    return (torch.clamp(torch.floor(G / s + 0.5), -8, 7) * s).reshape(W.shape)


def _lin64(x, W, tensor=False):
    q, s = _q64(x, tensor)
    return (q * s) @ W.t()


def _act64(y, act):
    return torch.relu(y) if act == "relu" else y / (1 + torch.exp(-y)) if act == "silu" else y


def exact(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        h = inp["x"].double()
        for i, W in enumerate(inp["W"]):
            h = _act64(_lin64(h, _w64(W), tensor=True), "relu" if i < 2 else "none")
        return h
    if kind == "decode":
        W = {k: _w64(w) for k, w in inp["W"].items()}
        o = _lin64(inp["attn"], W["o"])
        gu = _lin64(o, W["gate_up"])
        h = _act64(gu[:, :case["ff"]], "silu") * gu[:, case["ff"]:]
        return {"qkv": _lin64(inp["x"], W["qkv"]), "o": o, "gate_up": gu, "hq": None, "sh": _q64(h)[1].reshape(-1),
                "down": _lin64(h, W["down"])}
    if kind == "linear":
        y = _lin64(inp["x"], _w64(inp["W"]))
        if inp["bias"] is not None:
            y = y + inp["bias"].double()
        return (_act64(y, case["act"]), None, _q64(inp["x"])[1].reshape(-1))
    if kind == "prefill":
        W = inp["W"]
        qkv = _lin64(inp["X"], _w64(W["qkv"]))
        v = qkv[:, 8192:]
        o = _lin64(v, _w64(W["o"]))
        g, u = _lin64(o, _w64(W["gate"])), _lin64(o, _w64(W["up"]))
        h = _act64(g, "silu") * u
        return {"xq": None, "sx": _q64(inp["X"])[1].reshape(-1), "qkv": qkv, "vq": None, "sv": _q64(v)[1].reshape(-1),
                "o": o, "gate": g, "up": u, "oq": None, "so": _q64(o)[1].reshape(-1), "hq": None,
                "sh": _q64(h)[1].reshape(-1), "down": _lin64(h, _w64(W["down"]))}
    if kind == "quant":
        q, s = _q64(inp["x"])
        return (None, s.reshape(-1), q * s)
    if kind == "conv":
        x, w = inp["x"].double() - case["zp"], inp["w"].double()
        n, k, g = case["n"], case["k"], case["groups"]
        cg, og = case["c"] // g, case["o"] // g
        ho = (case["h"] + 2 * case["pad"] - k) // case["stride"] + 1
        wo = (case["w"] + 2 * case["pad"] - k) // case["stride"] + 1
        out = torch.empty((n, case["o"], ho * wo), dtype=torch.float64, device=DEV)
        for i in range(n):
            for j in range(g):
                col = F.unfold(x[i:i + 1, j * cg:(j + 1) * cg], k, padding=case["pad"], stride=case["stride"])[0]
                out[i, j * og:(j + 1) * og] = w[j * og:(j + 1) * og].reshape(og, -1) @ col
        return (out * inp["s_out"]).reshape(n, case["o"], ho, wo)
    if kind == "w4":
        W = {k: _w64(w, case["group"]) for k, w in inp["W"].items()}
        gu = _lin64(inp["x"], W["gate_up"])
        h = _act64(gu[:, :case["ff"]], "silu") * gu[:, case["ff"]:]
        return {"xq": None, "sx": _q64(inp["x"])[1].reshape(-1), "gate_up": gu, "hq": None,
                "sh": _q64(h)[1].reshape(-1), "down": _lin64(h, W["down"])}
    return None      # int32 sums

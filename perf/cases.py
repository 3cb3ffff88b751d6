"""The calls whose speed this repository watches, and how each is made, run and checked.

A case is one use of the W4A16 library through its Python binding: decode steps and verify rows
over the FFN layers of a model (captured into a HIP graph once, as a serving loop does), batches of
decoding sequences, single linears, and the load-time path that quantizes a weight, re-lays it into
tile order and reads it back. Weights are BF16 ~N(0, 0.02) quantized to symmetric INT4 in groups of
128, activations BF16 ~N(0, 1).

Ranges that the cases stand for: hidden 1024..5120 and intermediate 2048..17408, both any multiple
of 128; 1..128 activation rows; plain, RMSNorm, residual + RMSNorm (plan F2) and FP32-partial forms;
one layer called eagerly, or up to 64 in a graph.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "haskell-infer-demo_amd"))

import w4a16  # noqa: E402

GROUP = 128
EPS = 1e-6


def listed():
    return [
        # one projection of one token, called by itself: latency and launch cost
        dict(name="linear-decode", entry="linear", rows=1, k=2560, n=9728, layers=1, graph=False),
        # one decode token through the FFN half of every layer of a Qwen3-4B-shaped model, with the
        # residual updates and the norm that stand around it
        dict(name="decode-4b", entry="f2", rows=1, hidden=2560, inter=9728, layers=36, graph=True, style=1),
        # one decode token through 64 27B-class FFNs: the weight stream far past the caches
        dict(name="decode-27b", entry="mlp", rows=1, hidden=5120, inter=17408, layers=64, graph=True),
        # the same model on one of two tensor-parallel ranks: FP32 partials to be summed across ranks
        dict(name="decode-27b-tp2", entry="norm_partial", rows=1, hidden=5120, inter=8704, layers=16, graph=True,
             style=0),
        # a few speculative tokens verified at once
        dict(name="verify-4b", entry="norm", rows=4, hidden=2560, inter=9728, layers=36, graph=True, style=1),
        # the most rows a store routes to INT4
        dict(name="verify-27b", entry="f2", rows=16, hidden=5120, inter=17408, layers=16, graph=True,
             style=0),
        # a model whose sizes are odd numbers of groups, and an odd number of rows
        dict(name="verify-odd", entry="mlp", rows=7, hidden=3200, inter=8576, layers=24, graph=True),
        # one projection for a batch of sequences, from the M sweep of the single linear
        dict(name="linear-batch", entry="linear", rows=64, k=5120, n=4096, layers=24, graph=True),
        # a large batch of decoding sequences through every layer
        dict(name="batch-4b", entry="mlp", rows=128, hidden=2560, inter=9728, layers=36, graph=True),
        # a ragged batch, one layer called by itself
        dict(name="batch-27b-ragged", entry="norm", rows=50, hidden=5120, inter=17408, layers=1, graph=False,
             style=0),
        # load time: a gate/up pair quantized on the device and re-laid into tile order
        dict(name="quantize", entry="quantize", k=2560, n=19456, pair=True),
        # the check of a re-laid weight: back to FP32 rows
        dict(name="dequantize", entry="dequantize", k=9728, n=2560, pair=False),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    entry = rng.choice(["linear", "mlp", "mlp", "norm", "norm", "f2", "f2", "partial", "norm_partial", "quantize",
                        "dequantize"])
    hidden = 128 * round(_log_uniform(rng, 8, 40))
    inter = 128 * round(_log_uniform(rng, 16, 136))
    if entry in ("quantize", "dequantize"):
        pair = rng.random() < 0.5
        return dict(entry=entry, k=hidden, n=(2 if pair else 1) * (inter + 8 * rng.randrange(16)), pair=pair)
    rows = 1 if rng.random() < 0.3 else round(_log_uniform(rng, 1.5, 128))
    graph = rng.random() < 0.75
    if entry == "linear":
        k, n = (hidden, inter + 8 * rng.randrange(16)) if rng.random() < 0.5 else (inter, hidden)
        layers = rng.randint(8, 36) if graph else 1
        return dict(entry=entry, rows=rows, k=k, n=n, layers=layers, graph=graph)
    # no more work than the largest batch above
    most = 128 * 36 * 3 * 2560 * 9728 // (rows * 3 * hidden * inter)
    layers = min(rng.randint(4, 24), most) if graph else 1
    return dict(entry=entry, rows=rows, hidden=hidden, inter=inter, layers=layers, graph=graph,
                style=rng.randrange(2))


# ------------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------------


def _shapes(case):
    """[(n, k, pair)] of one layer's weights."""
    if case["entry"] in ("quantize", "dequantize"):
        return [(case["n"], case["k"], case["pair"])]
    if case["entry"] == "linear":
        return [(case["n"], case["k"], False)]
    h, i = case["hidden"], case["inter"]
    return [(2 * i, h, True), (h, i, False)]


def _weight(gen, n, k):
    """A checkpoint's BF16 weight, as FP32."""
    w = torch.empty(n, k, device="cuda").normal_(0.0, 0.02, generator=gen)
    return w.to(torch.bfloat16).float()


def _generators(seed):
    """One for the weights and one for everything else, so that exact() can make either alone."""
    gens = []
    for s in (2 * seed, 2 * seed + 1):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(s)
        gens.append(gen)
    return gens


def _activations(case, gen):
    """x (or the residual), the sublayer's output and the norm weight of every layer."""
    layers, rows = case["layers"], case["rows"]
    width = case["k"] if case["entry"] == "linear" else case["hidden"]

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    x = normal(layers, rows, width).to(torch.bfloat16)
    sub = normal(layers, rows, width).to(torch.bfloat16)
    # style 0 (Gemma) multiplies by 1 + weight, style 1 by the weight
    norm_w = (case.get("style", 0) + 0.1 * normal(layers, width)).to(torch.bfloat16)
    return x, sub, norm_w


def _tiled(w, n, k, pair):
    packed, scales = w4a16.quantize_device(w)
    return w4a16.TiledWeight.from_device_artifact(packed, scales, n, k, pair=pair)


def prepare(case, seed):
    wgen, xgen = _generators(seed)
    entry = case["entry"]
    if entry in ("quantize", "dequantize"):
        (n, k, pair), = _shapes(case)
        w = _weight(wgen, n, k)
        if entry == "quantize":
            return {"case": case, "w": w}
        return {"case": case, "tiled": _tiled(w, n, k, pair)}
    weights = [[_tiled(_weight(wgen, n, k), n, k, pair) for n, k, pair in _shapes(case)]
               for _ in range(case["layers"])]
    x, sub, norm_w = _activations(case, xgen)
    layers, rows = case["layers"], case["rows"]
    cols = case["n"] if entry == "linear" else case["hidden"]
    partial = entry in ("partial", "norm_partial")
    state = {"case": case, "weights": weights, "x": x, "sub": sub, "norm_w": norm_w}
    state["out"] = torch.empty(layers, rows, cols, device="cuda", dtype=torch.float32 if partial else torch.bfloat16)
    if entry == "f2":
        state["residual"] = torch.empty_like(x)
    if entry != "linear":
        ws_cols = case["inter"] if entry in ("mlp", "partial") else case["hidden"] + case["inter"]
        state["ws"] = torch.empty(rows, ws_cols, device="cuda", dtype=torch.bfloat16)
    if case["graph"]:
        # as a serving loop: one eager pass (first calls may allocate), then the capture
        _layers(state)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            _layers(state)
        torch.cuda.synchronize()
    return state


# ------------------------------------------------------------------------------------------------
# A pass
# ------------------------------------------------------------------------------------------------


def _layers(state):
    entry, style = state["case"]["entry"], state["case"].get("style", 0)
    x, out = state["x"], state["out"]
    if entry == "f2":
        state["residual"].copy_(x)  # updated in place below
    for i, w in enumerate(state["weights"]):
        if entry == "linear":
            w4a16.gemm_int4_bf16(x[i], w[0], out[i])
        elif entry in ("mlp", "partial"):
            w4a16.mlp_int4(x[i], w[0], w[1], out=out[i], act_ws=state["ws"], partial_f32=entry == "partial")
        elif entry in ("norm", "norm_partial"):
            w4a16.mlp_int4_norm(x[i], state["norm_w"][i], style, EPS, w[0], w[1], out=out[i], ws=state["ws"],
                                partial_f32=entry == "norm_partial")
        else:
            w4a16.mlp_int4_residual_norm(state["residual"][i], state["sub"][i], state["norm_w"][i], style, EPS, w[0],
                                         w[1], out=out[i], ws=state["ws"])


def run(state):
    case = state["case"]
    if case["entry"] == "quantize":
        packed, scales = w4a16.quantize_device(state["w"])
        tiled = w4a16.TiledWeight.from_device_artifact(packed, scales, case["n"], case["k"], pair=case["pair"])
        return {"packed": packed, "scales": scales, "tiled": tiled.packed, "tiled_scales": tiled.scales}
    if case["entry"] == "dequantize":
        return state["tiled"].dequantize()
    if case["graph"]:
        state["graph"].replay()
    else:
        _layers(state)
    if case["entry"] == "f2":
        return {"out": state["out"], "residual": state["residual"]}
    return state["out"]


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without, and what it is held to
# ------------------------------------------------------------------------------------------------


def work(case):
    shapes = _shapes(case)
    codes = sum(n * k // 2 + n * (k // GROUP) * 2 for n, k, _ in shapes)
    elems = sum(n * k for n, k, _ in shapes)
    if case["entry"] == "quantize":  # the weight in, the artifact and its tile order out
        return {"bytes": 4 * elems + 2 * codes, "flops": 3 * elems}
    if case["entry"] == "dequantize":
        return {"bytes": codes + 4 * elems, "flops": elems}
    rows, layers = case["rows"], case["layers"]
    if case["entry"] == "linear":
        io = rows * (case["k"] + case["n"]) * 2
    else:
        h = case["hidden"]
        io = rows * h * (2 + (4 if "partial" in case["entry"] else 2))
        if case["entry"] in ("norm", "norm_partial", "f2"):
            io += h * 2
        if case["entry"] == "f2":  # the sublayer in, the residual out
            io += 2 * rows * h * 2
    return {"bytes": layers * (codes + io), "flops": layers * 2 * rows * elems}


def tolerance(case):
    entry = case["entry"]
    if entry in ("quantize", "dequantize"):
        return "exact"
    # four times what the same rows differ by between row counts, which sum in other orders
    if entry in ("partial", "norm_partial"):
        # FP32 out of a BF16 intermediate, where a rounding that falls the other way moves it: 9.3e-5, 5e-4
        return {"rel": 4e-4, "max": 2e-3}
    # BF16 out, one ulp of which is 2^-8 of a value: 4.5e-5 for a linear, 5.2e-4 after a BF16
    # intermediate, 7.8e-3 at most
    return {"rel": 2e-4 if entry == "linear" else 2e-3, "max": 0.03}


def _bf16(v):
    return v.to(torch.float32).to(torch.bfloat16).double()


def _quantized(w):
    """(codes, scales) of an FP32 [n, k] weight: the format's rule, scale = BF16(absmax / 7)."""
    n, k = w.shape
    g = w.view(n, k // GROUP, GROUP)
    peak = g.abs().amax(-1)
    scales = torch.where(peak > 0, peak / 7.0, torch.ones_like(peak)).to(torch.bfloat16)
    codes = torch.clamp(torch.round(g / scales.float()[..., None]), -7, 7)
    return codes, scales


def _dequantized(w):
    n, k = w.shape
    codes, scales = _quantized(w)
    return (codes.double() * scales.double()[..., None]).view(n, k)


def exact(case, seed):
    if case["entry"] in ("quantize", "dequantize"):
        if case["entry"] == "quantize":
            return None  # whole numbers, compared as they are
        (n, k, _), = _shapes(case)
        return _dequantized(_weight(_generators(seed)[0], n, k))
    wgen, xgen = _generators(seed)
    entry = case["entry"]
    x, sub, norm_w = _activations(case, xgen)
    outs, residuals = [], []
    for i in range(case["layers"]):
        ws = [_dequantized(_weight(wgen, n, k)) for n, k, _ in _shapes(case)]
        v = x[i].double()
        if entry == "linear":
            outs.append(v @ ws[0].T)
            continue
        if entry == "f2":
            v = _bf16(v + sub[i].double())
            res = v
        if entry in ("norm", "norm_partial", "f2"):
            rms = torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS)
            v = _bf16(v * rms * (norm_w[i].double() + (1.0 - case["style"])))
        gate, up = _bf16(v @ ws[0].T).chunk(2, -1)
        act = _bf16(gate / (1.0 + torch.exp(-gate)) * up)
        outs.append(act @ ws[1].T)
        if entry == "f2":
            residuals.append(res + _bf16(outs[-1]))
    if entry == "f2":
        return {"out": torch.stack(outs), "residual": torch.stack(residuals)}
    return torch.stack(outs)

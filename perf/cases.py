"""The calls a user of the FP8 linear path makes, as measurable cases.

The sizes are the 9B projections of jeeves_amd/synthetic.py (hidden 4096, intermediate 12288, q/k/v merged to 6144,
lm_head 248320 rows, rank-16 LoRA), the batch sizes of bench.py (decode 1-128 rows, prefill 512-8192 tokens) and, in
draw(), generic multiples of 128 around them with odd row counts.

A case is one of these kinds:

linear   FP8Linear.forward, called eagerly (one projection, or the lm_head over the vocabulary)
matmul   fp8_matmul on row-major codes with a bias: the function form that the reference's callers use
mlp      FP8SwiGLU.forward, called eagerly
layer    one decoder layer's linears: the merged q/k/v projection, o and the SwiGLU block. With "graph" the three
         forward calls are captured once and replayed, as the engine replays its decode passes; the layer's weights
         are its own, so several layers in turn read them from HBM. With "lora" q, k, v, o, gate+up and down carry a
         rank-16 adapter each (q, k and v then stay apart). "act" is the arithmetic: "fp8", or "bf16" (the W8A16
         parity mode)
load     FP8Linear.load_weight: the quantization of a checkpoint's bf16 or fp32 weight, the row-major codes and the
         tiled copy that the kernels read
"""

import math

import torch

from jeeves_amd.fp8 import FP8Linear, FP8SwiGLU, fp8_matmul
from jeeves_amd.fp8_weights import quantize_rows

HIDDEN, INTER, QKV, KV, VOCAB = 4096, 12288, 6144, 1024, 248320
RANK, LORA_SCALING = 16, 2.0
FP8_MAX_RECIPROCAL = float(torch.tensor(1 / 448, dtype=torch.float32))


def _layer(name, m, act="fp8", graph=False, lora=False):
    return {"name": name, "kind": "layer", "m": m, "hidden": HIDDEN, "inter": INTER, "qkv": QKV, "act": act,
            "graph": graph, "lora": lora}


def listed():
    return [
        # one token through the narrowest projection, eagerly: the smallest call, host path and launches
        {"name": "linear_kv_m1", "kind": "linear", "m": 1, "n": KV, "k": HIDDEN, "act": "fp8"},
        # a decode step of one sequence
        _layer("decode_layer_m1", 1, graph=True),
        # a speculative block, or sixteen sequences: bench.py's headline step
        _layer("decode_layer_m16", 16, graph=True),
        # a full decode batch
        _layer("decode_layer_m64", 64, graph=True),
        # the logits of a few sequences
        {"name": "lm_head_m4", "kind": "linear", "m": 4, "n": VOCAB, "k": HIDDEN, "act": "fp8"},
        # a prompt of 2048 tokens
        _layer("prefill_layer_m2048", 2048),
        # many packed prompts of uneven lengths through the SwiGLU block: the largest call
        {"name": "mlp_m7921", "kind": "mlp", "m": 7921, "hidden": HIDDEN, "inter": INTER, "act": "fp8"},
        # a short prompt with an adapter on every projection
        _layer("lora_layer_m512", 512, lora=True),
        # the function form: row-major codes, a bias, an output width that is no whole tile
        {"name": "matmul_m333_n5000", "kind": "matmul", "m": 333, "n": 5000, "k": 2560, "bias": True},
        # the parity mode: decode and prefill in the reference's own arithmetic
        _layer("w8a16_layer_m32", 32, act="bf16", graph=True),
        _layer("w8a16_layer_m1024", 1024, act="bf16"),
        # a checkpoint's gate+up weight taken in
        {"name": "load_gate_up_bf16", "kind": "load", "n": 2 * INTER, "k": HIDDEN, "dtype": "bf16"},
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["linear", "matmul", "mlp", "layer", "layer", "layer", "layer", "load"])
    act = "bf16" if rng.random() < 0.2 else "fp8"
    sizes = [(4096, 12288, 6144), (128 * rng.randint(8, 40), 128 * rng.randint(24, 100), 16 * rng.randint(64, 640))]
    hidden, inter, qkv = rng.choice(sizes)
    if kind == "linear":
        n, k = rng.choice([(4096, 4096), (1024, 4096), (10240, 4096), (4096, 12288), (qkv, hidden), (VOCAB, 4096)])
        return {"kind": kind, "m": _between(rng, 1, 64 if n == VOCAB else 8192), "n": n, "k": k, "act": act}
    if kind == "matmul":
        return {"kind": kind, "m": _between(rng, 1, 4096), "n": _between(rng, 200, 20000), "k": 128 * _between(rng, 2, 64),
                "bias": rng.random() < 0.5}
    if kind == "load":
        return {"kind": kind, "n": 16 * _between(rng, 64, 1536), "k": 256 * _between(rng, 2, 48),
                "dtype": rng.choice(["bf16", "fp32"])}
    if kind == "mlp":
        return {"kind": kind, "m": _between(rng, 1, 6000 if act == "fp8" else 3000), "hidden": hidden, "inter": inter, "act": act}
    # decode steps are replayed as graphs, prompts run eagerly
    decode = rng.random() < 0.6
    m = _between(rng, 1, 128) if decode else _between(rng, 129, 3072 if act == "fp8" else 1536)
    lora = act == "fp8" and rng.random() < 0.25
    return {"kind": kind, "m": m, "hidden": hidden, "inter": inter, "qkv": qkv, "act": act, "graph": decode, "lora": lora}


def _shapes(case):
    """(name, n, k, the LoRA adapter's) of a case's linears."""
    kind = case["kind"]
    if kind in ("linear", "matmul", "load"):
        return [("w", case["n"], case["k"], False)]
    d, i, lora = case["hidden"], case["inter"], case.get("lora", False)
    mlp = [("gate_up", 2 * i, d, lora), ("down", d, i, lora)]
    if kind == "mlp":
        return mlp
    kv = case["qkv"] // 6 // 16 * 16
    qkv = [("q", case["qkv"] - 2 * kv, d, lora), ("k", kv, d, lora), ("v", kv, d, lora)] if lora else [("qkv", case["qkv"], d, False)]
    return qkv + [("o", d, d, lora)] + mlp


def _inputs(case, seed):
    """The bf16 activations, weights and adapters of a case, from the seed alone. Activations ~ N(0, 1) with eight
    outlier channels scaled x20 (up to 64 rows) or 1 % of the channels heavy-tailed; weights ~ N(0, 0.02)."""
    g = torch.Generator("cuda").manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dtype).mul_(std)

    def activations(m, k):
        x = normal(m, k, dtype=torch.float32)
        channels = torch.randperm(k, generator=g, device="cuda")
        if m <= 64:
            x[:, channels[:8]] *= 20.0
        else:
            c = channels[:max(1, k // 100)]
            chi = torch.randn(3, m, c.numel(), generator=g, device="cuda").pow_(2).sum(0) / 3.0
            x[:, c] = x[:, c] / chi.sqrt_()
        return x.to(torch.bfloat16)

    kind = case["kind"]
    wtype = torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16
    weights = {name: normal(n, k, std=0.02, dtype=wtype) for name, n, k, _ in _shapes(case)}
    lora = {name: (normal(RANK, k, std=0.01), normal(n, RANK, std=0.01)) for name, n, k, has in _shapes(case) if has}
    bias = normal(case["n"]) if case.get("bias") else None
    width = case["k"] if kind in ("linear", "matmul", "load") else case["hidden"]
    xs = [] if kind == "load" else [activations(case["m"], width) for _ in range(3 if kind == "layer" else 1)]
    return xs, weights, lora, bias


def _linear(weight, lora, act):
    m = FP8Linear(weight.shape[1], weight.shape[0], device="cuda")
    m.load_weight(weight)
    if lora is not None:
        m.set_lora(*lora, LORA_SCALING)
    m.set_activations(act)
    return m


def _forward(state):
    """The framework's calls for one pass, in order."""
    kind, xs, mods = state["kind"], state["xs"], state["mods"]
    if kind == "matmul":
        return [fp8_matmul(xs[0], state["codes"], state["scale"], bias=state["bias"])]
    if kind == "linear":
        return [mods["w"](xs[0])]
    if kind == "mlp":
        return [mods["mlp"](xs[0])]
    if kind == "load":
        mods["w"].load_weight(state["weight"])
        return [mods["w"].weight.view(torch.uint8), mods["w"].scale, mods["w"].kernel_weight()[0].view(torch.uint8)]
    return [mods[name](xs[0]) for name in ("q", "k", "v", "qkv") if name in mods] + [mods["o"](xs[1]), mods["mlp"](xs[2])]


_STREAM = []


def _capture(state):
    """One pass captured into a graph on a stream of its own, after an eager pass there (as warm() does before the
    engine captures)."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    s = _STREAM[0]
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        _forward(state)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            outs = _forward(state)
    torch.cuda.current_stream().wait_stream(s)
    return graph, outs


@torch.no_grad()
def prepare(case, seed):
    xs, weights, lora, bias = _inputs(case, seed)
    kind, act = case["kind"], case.get("act", "fp8")
    state = {"kind": kind, "xs": xs, "mods": {}, "graph": None}
    if kind == "load":
        state["weight"] = weights["w"]
        state["mods"]["w"] = FP8Linear(case["k"], case["n"], device="cuda")
        return state
    if kind == "matmul":
        state["codes"], state["scale"] = quantize_rows(weights["w"])
        state["bias"] = bias
        return state
    mods = {name: _linear(weights.pop(name), lora.get(name), act) for name, _, _, _ in _shapes(case)}
    if kind != "linear":
        mods["mlp"] = FP8SwiGLU(mods.pop("gate_up"), mods.pop("down"))
    state["mods"] = mods
    if case.get("graph"):
        state["graph"] = _capture(state)
    return state


@torch.no_grad()
def run(state):
    if state["graph"] is not None:
        graph, outs = state["graph"]
        graph.replay()
        return outs
    return _forward(state)


def work(case):
    """Codes, scales, adapters and activations read once, outputs written once; 2mnk per linear. h stays inside the
    SwiGLU block. A load reads the weight and writes both copies of the codes and the scales."""
    if case["kind"] == "load":
        n, k = case["n"], case["k"]
        return {"bytes": n * k * ((4 if case["dtype"] == "fp32" else 2) + 2) + 4 * n, "flops": 0}
    m, total, flops = case["m"], 0, 0
    for name, n, k, has in _shapes(case):
        total += n * k + 4 * n + (2 * n if case.get("bias") else 0)
        total += 0 if name in ("down", "k", "v") else 2 * m * k
        total += 0 if name == "gate_up" else 2 * m * n
        flops += 2 * m * n * k
        if has:
            total += 2 * RANK * (n + k)
            flops += 2 * m * RANK * (n + k)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Codes and scales of a load are the reference quantizer's, bit for bit. A linear's outputs are sums of exact
    products rounded once to bf16: measured 1.7e-3 from 64 bits, and one bf16 step of 2^-8 where two correct sums fall
    on the two sides of a tie. In a SwiGLU block such steps in gate and up move h and, with "fp8", some of h's codes
    by one: measured up to 5.4e-3 from 64 bits with outlier channels. Stated is about four times that."""
    if case["kind"] == "load":
        return "exact"
    if case["kind"] in ("linear", "matmul") or case["act"] == "bf16":
        return {"rel": 0.007, "max": 0.03}
    return {"rel": 0.02, "max": 0.3}


def _quantize(w):
    """(codes as float64, scale as float64) by the reference quantizer's definition, in plain torch."""
    w = w.float()
    scale = w.abs().amax(1).clamp_(min=1e-12) * FP8_MAX_RECIPROCAL
    codes = torch.empty(w.shape, dtype=torch.float8_e4m3fn, device=w.device)
    for r in range(0, w.shape[0], 16384):
        codes[r:r + 16384].view(torch.uint8).copy_((w[r:r + 16384] / scale[r:r + 16384, None]).to(torch.float8_e4m3fn).view(torch.uint8))
    return codes, scale


def _exact_linear(x, weight, lora, bias, act):
    codes, sw = _quantize(weight)
    a, sx = (x, None) if act == "bf16" else _quantize(x)
    y = torch.empty(x.shape[0], weight.shape[0], dtype=torch.float64, device=x.device)
    a = a.double()
    for r in range(0, weight.shape[0], 16384):
        y[:, r:r + 16384] = a @ codes[r:r + 16384].double().t().contiguous()
    y *= sw.double()
    if sx is not None:
        y *= sx.double()[:, None]
    if lora is not None:
        y += LORA_SCALING * ((x.double() @ lora[0].double().t().contiguous()) @ lora[1].double().t().contiguous())
    if bias is not None:
        # the bias is added to the linear's bf16 output
        y = y.to(torch.bfloat16).double() + bias.double()
    return y


def _exact_mlp(x, weights, lora, act):
    gu = _exact_linear(x, weights["gate_up"], lora.get("gate_up"), None, act).to(torch.bfloat16)
    gate, up = gu.chunk(2, dim=1)
    # F.silu(gate) * up on bf16 tensors: silu rounded, then the product
    h = (torch.nn.functional.silu(gate.double()).to(torch.bfloat16).double() * up.double()).to(torch.bfloat16)
    return _exact_linear(h, weights["down"], lora.get("down"), None, act)


@torch.no_grad()
def exact(case, seed):
    xs, weights, lora, bias = _inputs(case, seed)
    kind, act = case["kind"], case.get("act", "fp8")
    if kind == "load":
        codes, scale = _quantize(weights["w"])
        n, k = codes.shape
        codes = codes.view(torch.uint8)
        # the tiled copy: 16 rows by 128 columns a tile, halves of 16 columns interleaved
        tiled = codes.view(n // 16, 16, k // 128, 4, 2, 16).permute(0, 2, 4, 3, 1, 5).reshape(n, k)
        return [codes, scale, tiled]
    if kind in ("linear", "matmul"):
        return [_exact_linear(xs[0], weights["w"], None, bias, act)]
    if kind == "mlp":
        return [_exact_mlp(xs[0], weights, lora, act)]
    first = [_exact_linear(xs[0], weights[name], lora.get(name), None, act) for name in ("q", "k", "v", "qkv") if name in weights]
    return first + [_exact_linear(xs[1], weights["o"], lora.get("o"), None, act), _exact_mlp(xs[2], weights, lora, act)]

"""What a program does with this package, as cases that can be measured.

The package is the W8A8 int8 path of an LLM server: the scaled matmul with vLLM's scaled_mm
contract, the activation quantizers around it, and the two composed into decoder layers.  A
case names one such call, its sizes and its options:

  linear   w8a8_mm over one projection: decode (few tokens), batched decode, chunked and full
           prefill; the Qwen3-1.7B and Llama-3-8B projections, and generic sizes (other hidden
           and MLP widths, tensor-parallel shards) that the library has no tuned entry for;
           per-token or one activation scale, bf16 / fp16 / fp32 output, with and without bias
  norm     add_rmsnorm_quant: the residual add, RMSNorm and quantizer in front of a projection
  silu     silu_mul_quant: the MLP's activation and quantizer in front of down_proj
  quant    quant_per_token over the query columns of a qkv output, read in place
  step     the 28-layer Qwen3-1.7B decoder stand-in's decode step for a batch of sequences,
           captured once as a HIP graph and replayed for each token, as a server runs it
  prefill  one decoder layer of the same stand-in over a prompt, called eagerly
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "int8-linear_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from int8_linear import standin, w8a8_mm  # noqa: E402
from int8_linear import fused_quant as fq  # noqa: E402

DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
DECODE_LAYERS = 28   # the model's depth
PREFILL_LAYERS = 1

# (K, N) of the projections of the two models the benchmark runs, merged as a server runs them
QWEN = [(2048, 4096), (2048, 2048), (2048, 12288), (6144, 2048)]
LLAMA = [(4096, 6144), (4096, 4096), (4096, 28672), (14336, 4096)]
# generic: other hidden and MLP widths, and the shards of a tensor-parallel split
GENERIC = [(5120, 7680), (5120, 5120), (13824, 5120), (3584, 4608), (3584, 18944),
           (8192, 10240), (4096, 1536), (1792, 4096), (2560, 9728), (1024, 4096),
           (4096, 5504), (2752, 4096)]
HIDDEN = [1024, 2048, 2560, 3584, 4096, 5120, 8192]
MLP = [1536, 1792, 3072, 6144, 8960, 9728, 13824, 14336, 18944]

MAX_FLOPS = 2.0 * 4096 * 4096 * 28672  # the largest listed case's


def listed():
    return [
        # one sequence's token through the smallest merged projection: launch and latency
        {"name": "linear qkv 1", "kind": "linear", "m": 1, "k": 2048, "n": 4096,
         "out": "bf16", "bias": False, "per_token": True},
        # a decode batch through the widest projection, with the bias some models carry
        {"name": "linear gate_up 24 bias", "kind": "linear", "m": 24, "k": 4096, "n": 28672,
         "out": "bf16", "bias": True, "per_token": True},
        # a ragged batch of sequences through the longest reduction
        {"name": "linear down 75", "kind": "linear", "m": 75, "k": 14336, "n": 4096,
         "out": "bf16", "bias": False, "per_token": True},
        # a ragged chunk of a prompt, an fp16 model with qkv bias
        {"name": "linear qkv 777 fp16 bias", "kind": "linear", "m": 777, "k": 4096, "n": 6144,
         "out": "fp16", "bias": True, "per_token": True},
        # sizes without a tuned entry, a static (per-tensor) activation scale, fp32 output
        {"name": "linear generic 1500 fp32", "kind": "linear", "m": 1500, "k": 5120, "n": 7680,
         "out": "fp32", "bias": False, "per_token": False},
        # a full prompt through the widest projection
        {"name": "linear gate_up 4096", "kind": "linear", "m": 4096, "k": 4096, "n": 28672,
         "out": "bf16", "bias": False, "per_token": True},
        # the norm in front of a projection, over a full prompt of the 4096-wide model
        {"name": "norm 4096 x 4096", "kind": "norm", "m": 4096, "h": 4096, "act": "bf16",
         "residual": True},
        # the MLP's activation over a ragged prompt, rounded as the served models do
        {"name": "silu 3001 x 14336", "kind": "silu", "m": 3001, "i": 14336, "act": "bf16",
         "round": True},
        # the query columns of a batch's qkv output, in front of o_proj
        {"name": "quant 512 x 4096", "kind": "quant", "m": 512, "h": 4096, "ld": 6144,
         "act": "bf16"},
        # decode: one sequence, and a ragged batch of them
        {"name": "step 1", "kind": "step", "m": 1},
        {"name": "step 100", "kind": "step", "m": 100},
        # prefill: a full prompt through a layer
        {"name": "prefill 4096", "kind": "prefill", "m": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], evenly spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "norm", "silu", "quant", "step", "prefill"])
    if kind == "linear":
        k, n = rng.choice(rng.choice([QWEN, LLAMA, GENERIC]))
        m = _log(rng, 1, min(8192, int(MAX_FLOPS / (2.0 * k * n))))
        return {"kind": kind, "m": m, "k": k, "n": n,
                "out": rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]),
                "bias": rng.random() < 0.4, "per_token": rng.random() < 0.85}
    act = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "norm":
        return {"kind": kind, "m": _log(rng, 1, 8192), "h": rng.choice(HIDDEN), "act": act,
                "residual": rng.random() < 0.8}
    if kind == "silu":
        return {"kind": kind, "m": _log(rng, 1, 4096), "i": rng.choice(MLP), "act": act,
                "round": rng.random() < 0.6}
    if kind == "quant":
        h = rng.choice(HIDDEN)
        return {"kind": kind, "m": _log(rng, 1, 8192), "h": h,
                "ld": rng.choice([h, h + h // 2, 2 * h]), "act": act}
    if kind == "step":
        return {"kind": kind, "m": _log(rng, 2, 99)}
    return {"kind": kind, "m": _log(rng, 129, 4095)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _quant_rows(x):
    """Symmetric int8 codes of each row and the row's fp32 scale."""
    scale = x.abs().amax(dim=1, keepdim=True).clamp_min(1e-8) / 127.0
    return (x / scale).round_().clamp_(-127, 127).to(torch.int8), scale


def _randn(shape, g, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        m, k, n, out = case["m"], case["k"], case["n"], DTYPE[case["out"]]
        x = _randn((m, k), g).to(torch.bfloat16).float()
        if case["per_token"]:
            a_q, a_s = _quant_rows(x)
        else:
            a_s = (x.abs().max() / 127.0).reshape(1)
            a_q = (x / a_s).round().clamp(-127, 127).to(torch.int8)
        w_q, w_s = _quant_rows(_randn((n, k), g, 0.02))
        bias = _randn((n,), g, 0.01).to(out) if case["bias"] else None
        return {"case": case, "a": a_q, "sa": a_s, "w": w_q.t(), "sb": w_s, "bias": bias, "out": out}
    if kind in ("step", "prefill"):
        layers = DECODE_LAYERS if kind == "step" else PREFILL_LAYERS
        stack = standin.DecoderStandIn(case["m"], layers, seed=int(seed), device="cuda",
                                       generator_device="cuda")
        state = {"case": case, "stack": stack}
        if kind == "step":
            # warm up once on a side stream, then capture the step, as a serving loop does
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                stack.forward(with_residual=True)
            torch.cuda.current_stream().wait_stream(side)
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                state["result"] = stack.forward(with_residual=True)
        return state
    act = DTYPE[case["act"]]
    if kind == "norm":
        shape = (case["m"], case["h"])
        res = _randn(shape, g, 2.0).to(act) if case["residual"] else None
        w = (1.0 + _randn((case["h"],), g, 0.1)).to(act)
        return {"case": case, "x": _randn(shape, g).to(act), "res": res, "w": w}
    if kind == "silu":
        return {"case": case, "x": _randn((case["m"], 2 * case["i"]), g, 2.0).to(act)}
    wide = _randn((case["m"], case["ld"]), g).to(act)
    return {"case": case, "x": wide[:, :case["h"]]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return w8a8_mm(state["a"], state["w"], state["sa"], state["sb"], state["out"], state["bias"])
    if kind == "step":
        state["graph"].replay()
        return state["result"]
    if kind == "prefill":
        return state["stack"].forward(with_residual=True)
    if kind == "norm":
        q, s, res = fq.add_rmsnorm_quant(state["x"], state["res"], state["w"], standin.EPS)
        return (q, s, res) if res is not None else (q, s)
    if kind == "silu":
        return fq.silu_mul_quant(state["x"], True, case["round"])
    return fq.quant_per_token(state["x"])


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "linear":
        k, n = case["k"], case["n"]
        b = m * k + k * n + BYTES[case["out"]] * m * n + 4 * (m if case["per_token"] else 1) + 4 * n
        b += BYTES[case["out"]] * n if case["bias"] else 0
        return {"bytes": b, "flops": 2.0 * m * k * n}
    if kind == "norm":
        h = case["h"]
        return {"bytes": (7 if case["residual"] else 3) * m * h + 2 * h + 4 * m, "flops": 0}
    if kind == "silu":
        return {"bytes": 5 * m * case["i"] + 4 * m, "flops": 0}
    if kind == "quant":
        return {"bytes": 3 * m * case["h"] + 4 * m, "flops": 0}
    layers = DECODE_LAYERS if kind == "step" else PREFILL_LAYERS
    per_layer = sum(k * n for k, n in QWEN)
    scales = sum(4 * n for _, n in QWEN)
    return {"bytes": layers * (per_layer + scales) + 3 * 2 * m * standin.HIDDEN,
            "flops": 2.0 * m * layers * per_layer}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        # an exact int32 product, then one rounding to the output type (measured against exact():
        # 1.7e-3 in bf16, 2.1e-4 in fp16, 6e-8 in fp32)
        return {"bf16": {"rel": 7e-3, "max": 1.6e-2}, "fp16": {"rel": 8e-4, "max": 2e-3},
                "fp32": {"rel": 1e-6, "max": 4e-6}}[case["out"]]
    if kind in ("step", "prefill"):
        # bf16 between the operations and int8 codes in front of every projection: a code that
        # falls the other way at a rounding boundary moves all that follows it
        return {"rel": 3e-2, "max": 2.5e-1}
    # scales to fp32 rounding; the residual stream to one rounding of its type; a code or a
    # 16-bit value on a rounding boundary may fall either way
    return {"rel": 7e-3, "max": 1.6e-2, "differ": 2e-3}


# ------------------------------------------------------------------ the same in 64 bits
def _codes(y):
    """Quantizer of 64-bit rows: codes and scale."""
    absmax = y.abs().amax(dim=1, keepdim=True)
    inv = torch.where(absmax > 0, 127.0 / absmax, torch.zeros_like(absmax))
    return (y * inv).round().clamp(-128, 127), absmax / 127.0


def _norm(s, w, act):
    y = s * torch.rsqrt((s * s).mean(dim=1, keepdim=True) + standin.EPS)
    return ((y.to(act)).double() * w.double()).to(act).double()


def _silu(x, act, rounded):
    i = x.shape[1] // 2
    g, u = x[:, :i].double(), x[:, i:].double()
    a = g * torch.sigmoid(g)
    a = a.to(act).double() if rounded else a
    return (a * u).to(act).double()


def _exact_layers(stack):
    res, h = None, stack.x.double()
    for layer in stack.layers:
        def mm(q, s, name):
            w, ws = layer[name]
            return ((q @ w.t().double()) * s * ws.reshape(1, -1).double()).to(torch.bfloat16).double()
        res = h if res is None else res + h
        q, s = _codes(_norm(res, stack.norm, torch.bfloat16))
        res = res.to(torch.bfloat16).double()
        q, s = _codes(mm(q, s, "qkv_proj")[:, :standin.Q_COLS])
        res = res + mm(q, s, "o_proj")
        q, s = _codes(_norm(res, stack.norm, torch.bfloat16))
        res = res.to(torch.bfloat16).double()
        q, s = _codes(_silu(mm(q, s, "gate_up_proj"), torch.bfloat16, fq.ROUND_SILU))
        h = mm(q, s, "down_proj")
    return h, res


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        # 28 layers of random weights amplify every code that falls the other way at a rounding
        # boundary until the chains are far apart: there is no 64-bit value to compare with
        return None
    if kind == "prefill":
        return _exact_layers(standin.DecoderStandIn(case["m"], PREFILL_LAYERS, seed=int(seed),
                                                    device="cuda", generator_device="cuda"))
    st = prepare(case, seed)
    if kind == "linear":
        c = (st["a"].double() @ st["w"].double()) * st["sa"].double().reshape(-1, 1)
        c = c * st["sb"].double().reshape(1, -1)
        return c + st["bias"].double() if st["bias"] is not None else c
    act = DTYPE[case["act"]]
    if kind == "norm":
        s = st["x"].double() + (st["res"].double() if st["res"] is not None else 0.0)
        q, scale = _codes(_norm(s, st["w"], act))
        return (q, scale, s) if st["res"] is not None else (q, scale)
    if kind == "silu":
        return _codes(_silu(st["x"], act, case["round"]))
    return _codes(st["x"].double())

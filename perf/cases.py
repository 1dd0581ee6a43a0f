"""The work a user of this library has it do, as cases that can be timed.

Every case goes through a public entry point: the layers of
``inference_systems_amd.layers`` with ``gemm_backend = "hip"``, the backend
switch ``linear`` and ``gemm_kn``.  Sizes are those of the Qwen3.5-0.8B
projections the layers mirror (hidden 1024, intermediate 3584, vocabulary
151936), of the reference's GEMM shape table, and generic ones between them.

A case is a dict of plain values:

  op      "linear"   linear(x[M, K], W[N, K])       "kn"     gemm_kn(x[M, K], B[K, N])
          "mlp"      Qwen35MLP.forward_add_norm      "gdn"    GdnInputProjection.forward_add_norm
          "gated"    RowParallelLinear.forward_gated
          "logits"   ParallelLMHead(x)               "sample" ParallelLMHead.sample
          "greedy"   ParallelLMHead.greedy
          "step"     the projections of a few decoder layers, captured once in a HIP graph and replayed
  dtype   input type ("bf16", "f16", "f32"); out: output type where the entry point lets the caller choose
  m, n, k sizes: n output columns (intermediate size for "mlp"), k the contraction (hidden size for "mlp")
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

PKG = __graft_entry__.load_package()
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EPS = 1e-6
HEAD_DIM = 128      # gate groups of the gated projection, and the value heads of "gdn"
STEP_LAYERS = 4     # decoder layers of a "step" case


def listed():
    return [
        # One token of one sequence through a projection: the smallest call a decode loop makes.
        {"name": "decode 1x6144x1024", "op": "linear", "dtype": "bf16", "out": "bf16", "m": 1, "n": 6144, "k": 1024},
        # Post-attention norm and MLP of a batched decode step, called eagerly.
        {"name": "decode mlp 16", "op": "mlp", "dtype": "bf16", "m": 16, "n": 3584, "k": 1024},
        # Output gate and o_proj of a small decode batch, called eagerly.
        {"name": "decode gated o_proj 4", "op": "gated", "dtype": "bf16", "m": 4, "n": 1024, "k": 2048},
        # Decode as a serving loop runs it: the layers' projections captured in one HIP graph.
        {"name": "decode step graph 32", "op": "step", "dtype": "bf16", "m": 32, "n": 3584, "k": 1024},
        # The sampled token of a decode batch from the tied LM head.
        {"name": "lm head sample 32", "op": "sample", "dtype": "bf16", "m": 32, "n": 151936, "k": 1024},
        # A short prompt or a prefill chunk through the MLP's down projection (a ragged token count).
        {"name": "chunk down 200x1024x3584", "op": "linear", "dtype": "bf16", "out": "bf16", "m": 200, "n": 1024,
         "k": 3584},
        # Prefill of 2048 tokens through a projection.
        {"name": "prefill 2048x4096x1024", "op": "linear", "dtype": "bf16", "out": "bf16", "m": 2048, "n": 4096,
         "k": 1024},
        # fp16 prefill through the long-K down projection.
        {"name": "prefill down f16", "op": "linear", "dtype": "f16", "out": "f16", "m": 4096, "n": 1024, "k": 3584},
        # Norm and MLP of a large prefill batch.
        {"name": "prefill mlp 8192", "op": "mlp", "dtype": "bf16", "m": 8192, "n": 3584, "k": 1024},
        # fp32 model code: a square product on B[K, N].
        {"name": "f32 square 1024 kn", "op": "kn", "dtype": "f32", "out": "f32", "m": 1024, "n": 1024, "k": 1024},
        # fp32 decode batch on a projection.
        {"name": "f32 decode 16x6144x1024", "op": "linear", "dtype": "f32", "out": "f32", "m": 16, "n": 6144,
         "k": 1024},
        # Sizes that are no multiple of anything.
        {"name": "odd 333x1001x1003", "op": "linear", "dtype": "bf16", "out": "f32", "m": 333, "n": 1001, "k": 1003},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size over the logarithm of [lo, hi]: mostly what weights have (multiples of 64), else any."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.3 else max(lo, (v + 32) // 64 * 64)


def draw(rng):
    op = rng.choice(["linear"] * 5 + ["kn"] * 2 + ["mlp"] * 2 + ["gated", "gdn", "logits", "sample", "greedy", "step"])
    half = rng.choice(["bf16", "bf16", "f16"])
    if op in ("linear", "kn"):
        dtype = rng.choice([half, half, half, "f32"])
        # fp32 and element-wise operands run at a fraction of the bf16 rate: the same time is less work.
        while True:
            m, n, k = _log(rng, 1, 8192), _size(rng, 64, 16384), _size(rng, 64, 8192)
            limit = 1e11 if dtype != "f32" and k % 8 == 0 and (op == "linear" or n % 8 == 0) else 1.2e10
            if 2.0 * m * n * k <= limit:
                break
        return {"op": op, "dtype": dtype, "out": rng.choice([dtype, "f32"]), "m": m, "n": n, "k": k}
    if op == "mlp":
        return {"op": op, "dtype": "bf16", "m": _log(rng, 1, 6000), "n": 64 * rng.randint(8, 64),
                "k": 64 * rng.randint(8, 24)}
    if op == "gated":
        return {"op": op, "dtype": half, "m": _log(rng, 1, 8192), "n": 64 * rng.randint(8, 40),
                "k": HEAD_DIM * rng.randint(4, 32)}
    if op == "gdn":
        return {"op": op, "dtype": "bf16", "m": _log(rng, 1, 4096), "n": rng.choice([4, 8, 16, 24]),
                "k": 64 * rng.randint(8, 24)}
    if op == "logits":
        return {"op": op, "dtype": half, "out": rng.choice([half, "f32"]), "m": _log(rng, 1, 400),
                "n": rng.randint(30000, 152000), "k": 64 * rng.randint(8, 20)}
    if op in ("sample", "greedy"):
        return {"op": op, "dtype": half, "m": _log(rng, 1, 300), "n": rng.randint(30000, 152000),
                "k": 64 * rng.randint(8, 20)}
    return {"op": "step", "dtype": "bf16", "m": rng.randint(1, 64), "n": 64 * rng.randint(16, 64),
            "k": 64 * rng.randint(8, 24)}


# ---------------------------------------------------------------------------
# Inputs.  Activations are standard normal, weights normal with deviation
# 0.02, norm weights small around their zero centre.
# ---------------------------------------------------------------------------
class _Inputs:
    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device=DEV).manual_seed(int(seed))
        self.dtype = dtype

    def normal(self, *shape, std=1.0):
        return (torch.randn(shape, generator=self.gen, device=DEV) * std).to(self.dtype)

    def weight(self, *shape):
        return self.normal(*shape, std=0.02)


def _load(layer, weight, dtype):
    """The layer with its weight in place, on the GPU, routed through the library."""
    layer.weight = torch.nn.Parameter(weight, requires_grad=False)
    layer = layer.to(DEV, dtype)
    layer.gemm_backend = "hip"
    return layer


def _norm(inp, hidden):
    norm = PKG.layers.Qwen35RMSNorm(hidden, EPS)
    norm.weight = torch.nn.Parameter(inp.normal(hidden, std=0.1), requires_grad=False)
    return norm.to(DEV)


def _mlp(inp, hidden, inter):
    with torch.device("meta"):
        mlp = PKG.layers.Qwen35MLP(hidden, inter)
    mlp.gate_up_proj.weight = torch.nn.Parameter(inp.weight(2 * inter, hidden), requires_grad=False)
    mlp.down_proj.weight = torch.nn.Parameter(inp.weight(hidden, inter), requires_grad=False)
    mlp.gemm_backend = "hip"
    return mlp


def _gdn(inp, hidden, heads):
    with torch.device("meta"):
        proj = PKG.layers.GdnInputProjection(hidden, heads, heads, HEAD_DIM, HEAD_DIM)
    rows = sum(proj.output_sizes)
    return _load(proj, inp.weight(rows, hidden), inp.dtype)


def _row_parallel(inp, k, n):
    with torch.device("meta"):
        layer = PKG.layers.RowParallelLinear(k, n)
    return _load(layer, inp.weight(n, k), inp.dtype)


def _gated_inputs(inp, m, k):
    """Attention output [M, heads, head_dim] and the gate half of q_proj's output."""
    heads = k // HEAD_DIM
    x = inp.normal(m, heads, HEAD_DIM)
    gate = inp.normal(m, heads, 2 * HEAD_DIM).chunk(2, -1)[1]
    return x, gate


def prepare(case, seed):
    op, m, n, k = case["op"], case["m"], case["n"], case["k"]
    dtype = DTYPES[case["dtype"]]
    inp = _Inputs(seed, dtype)
    s = {"op": op}
    with torch.inference_mode():
        if op == "linear":
            s.update(x=inp.normal(m, k), w=inp.weight(n, k), out=DTYPES[case["out"]])
        elif op == "kn":
            s.update(x=inp.normal(m, k), w=inp.weight(k, n), out=DTYPES[case["out"]])
        elif op == "mlp":
            s.update(h=inp.normal(m, k), r=inp.normal(m, k), norm=_norm(inp, k), layer=_mlp(inp, k, n))
        elif op == "gdn":
            s.update(h=inp.normal(m, k), r=inp.normal(m, k), norm=_norm(inp, k), layer=_gdn(inp, k, n))
        elif op == "gated":
            x, gate = _gated_inputs(inp, m, k)
            s.update(x=x, gate=gate, layer=_row_parallel(inp, k, n))
        elif op in ("logits", "sample", "greedy"):
            with torch.device("meta"):
                head = PKG.layers.ParallelLMHead(n, k)
            s.update(x=inp.normal(m, k), head=_load(head, inp.weight(n, k), dtype))
            if op == "logits":
                s["head"].logits_dtype = DTYPES[case["out"]]
            elif op == "sample":
                # Sampled rows at usual temperatures, and one in four greedy.
                t = 0.6 + 0.6 * torch.rand(m, generator=inp.gen, device=DEV)
                t[::4] = 0.0
                s.update(t=t, seed=int(seed) + 17, offset=3)
        else:
            _prepare_step(s, inp, m, n, k)
    return s


def _prepare_step(s, inp, m, n, k):
    """STEP_LAYERS decoder layers: norm and merged input projection, output
    gate and o_proj on the attention output (an input here: attention is not
    this library's), norm and MLP.  A serving loop captures this once and
    replays it for every token."""
    heads = max(1, k // HEAD_DIM)
    s.update(h=inp.normal(m, k), r=inp.normal(m, k), layers=[])
    for _ in range(STEP_LAYERS):
        x, gate = _gated_inputs(inp, m, heads * HEAD_DIM)
        s["layers"].append({"norm1": _norm(inp, k), "gdn": _gdn(inp, k, heads), "x": x, "gate": gate,
                            "o_proj": _row_parallel(inp, heads * HEAD_DIM, k), "norm2": _norm(inp, k),
                            "mlp": _mlp(inp, k, n)})
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(s)
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        s["outputs"] = _step(s)


def _step(s):
    h, r, parts = s["h"], s["r"], []
    for lay in s["layers"]:
        y, r = lay["gdn"].forward_add_norm(h, r, lay["norm1"])
        parts.append(y[0])
        h = lay["o_proj"].forward_gated(lay["x"], lay["gate"])
        h, r = lay["mlp"].forward_add_norm(h, r, lay["norm2"])
    return {"h": h, "r": r, "qkv": parts}


# ---------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------
@torch.inference_mode()
def run(s):
    op = s["op"]
    if op == "linear":
        return PKG.linear(s["x"], s["w"], out_dtype=s["out"], backend="hip")
    if op == "kn":
        return PKG.gemm_kn(s["x"], s["w"], s["out"])
    if op == "mlp":
        return s["layer"].forward_add_norm(s["h"], s["r"], s["norm"])
    if op == "gdn":
        y, r = s["layer"].forward_add_norm(s["h"], s["r"], s["norm"])
        return {"parts": list(y), "r": r}
    if op == "gated":
        return s["layer"].forward_gated(s["x"], s["gate"])
    if op == "logits":
        return s["head"](s["x"])
    if op == "sample":
        return s["head"].sample(s["x"], s["t"], s["seed"], s["offset"])
    if op == "greedy":
        return s["head"].greedy(s["x"])
    s["graph"].replay()
    return s["outputs"]


# ---------------------------------------------------------------------------
# What a pass cannot do without.
# ---------------------------------------------------------------------------
def work(case):
    op, m, n, k = case["op"], case["m"], case["n"], case["k"]
    size = 4 if case["dtype"] == "f32" else 2
    gemm = lambda m, n, k: 2.0 * m * n * k  # noqa: E731
    if op in ("linear", "kn", "logits"):
        return {"bytes": size * (m * k + n * k) + (4 if case["out"] == "f32" else 2) * m * n, "flops": gemm(m, n, k)}
    if op == "gated":
        return {"bytes": 2 * (2 * m * k + n * k + m * n), "flops": gemm(m, n, k)}
    if op in ("sample", "greedy"):
        return {"bytes": 2 * (m * k + n * k) + 12 * m, "flops": gemm(m, n, k)}
    mlp = {"bytes": 2 * (2 * m * k + 3 * n * k + 2 * m * k), "flops": gemm(m, 3 * n, k)}
    if op == "mlp":
        return mlp
    heads = n if op == "gdn" else max(1, k // HEAD_DIM)
    rows = heads * (4 * HEAD_DIM + 2)
    gdn = {"bytes": 2 * (2 * m * k + rows * k + m * rows + m * k), "flops": gemm(m, rows, k)}
    if op == "gdn":
        return gdn
    wide = heads * HEAD_DIM
    o_proj = {"bytes": 2 * (2 * m * wide + wide * k + m * k), "flops": gemm(m, k, wide)}
    return {key: STEP_LAYERS * (gdn[key] + o_proj[key] + mlp[key]) for key in ("bytes", "flops")}


def tolerance(case):
    """About four times what the outputs differ by from the same arithmetic
    on another GEMM (torch's), i.e. with sums in another order: fp32 outputs
    by up to 8e-7 in norm and 4e-6 in one value, fp16 by 2.4e-5 and 1e-3,
    bf16 by 5e-5 and 8e-3 (single values rounded the other way).  The norm's
    operand is rounded at another place there: 5.6e-3 after an MLP, 7.6e-3
    after four layers."""
    op = case["op"]
    if op == "step":
        return {"rel": 2e-2, "max": 0.15}
    if op in ("mlp", "gdn"):
        return {"rel": 1e-2, "max": 0.1}
    if op in ("sample", "greedy"):
        # The ranked logits are rounded to the input type: a row's winner changes only where two
        # candidates tie.
        return {"rel": 2e-3, "max": 0.03, "differ": 0.01}
    if op == "gated":
        return {"rel": 2e-3, "max": 0.03}
    if case["out"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 1e-3, "max": 0.03} if case["out"] == "bf16" else {"rel": 2e-4, "max": 4e-3}


# ---------------------------------------------------------------------------
# The same outputs in 64 bits.
# ---------------------------------------------------------------------------
def _exact_norm(h, r, norm):
    s = h.double() + r.double()
    scale = torch.rsqrt(s.square().mean(-1, keepdim=True) + EPS)
    return s * scale * (1.0 + norm.weight.double()), s


def _exact_mlp(h, r, norm, mlp):
    y, s = _exact_norm(h, r, norm)
    gate, up = (y @ mlp.gate_up_proj.weight.double().T).chunk(2, -1)
    return (gate * torch.sigmoid(gate) * up) @ mlp.down_proj.weight.double().T, s


def _exact_gated(x, gate, weight):
    return (x.double() * torch.sigmoid(gate.double())).reshape(x.shape[0], -1) @ weight.double().T


@torch.inference_mode()
def exact(case, seed):
    op = case["op"]
    if op == "sample":
        return None     # the draws are the library's own
    s = prepare(case, seed)
    if op == "linear":
        return s["x"].double() @ s["w"].double().T
    if op == "kn":
        return s["x"].double() @ s["w"].double()
    if op == "mlp":
        return _exact_mlp(s["h"], s["r"], s["norm"], s["layer"])
    if op == "gdn":
        y, r = _exact_norm(s["h"], s["r"], s["norm"])
        y = y @ s["layer"].weight.double().T
        return {"parts": list(y.split(s["layer"].output_sizes, -1)), "r": r}
    if op == "gated":
        return _exact_gated(s["x"], s["gate"], s["layer"].weight)
    if op in ("logits", "greedy"):
        logits = s["x"].double() @ s["head"].weight.double().T
        return logits if op == "logits" else (None, logits.max(-1).values)
    h, r, parts = s["h"], s["r"], []
    for lay in s["layers"]:
        y, r = _exact_norm(h, r, lay["norm1"])
        parts.append((y @ lay["gdn"].weight.double().T)[:, : lay["gdn"].conv_dim])
        h = _exact_gated(lay["x"], lay["gate"], lay["o_proj"].weight)
        h, r = _exact_mlp(h, r, lay["norm2"], lay["mlp"])
    return {"h": h, "r": r, "qkv": parts}

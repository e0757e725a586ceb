"""The workloads that this library's speed is judged by, through its public entry points.

Five kinds of pass, over the sizes that a caller meets between one decode row
and a long prefill:

* ``call``  -- one eager ``marlin.gemm_fast``, the per-token call;
* ``layer`` -- one dense decoder layer on INT4 Marlin weights: up to 16 rows
  the captured ``DecodeLayerGraph``, above the eager chain of a prefill or a
  large decode batch (norm, qkv, o, norm, gate/up, SwiGLU, down);
* ``fp8``   -- the three FP8 128x128-block linears of a dense layer, several
  layers in one captured graph up to 16 rows, eager above;
* ``moe``   -- one ``moe_branch`` (gate, routing, routed and shared experts) per
  layer, several layers in one captured graph up to 16 tokens, eager above.

Packing weights is left out: a program does it once, when it loads a model.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fastllm-py_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from fastllm_py.decode_graph import DecodeLayerGraph  # noqa: E402
from fastllm_py.kernels import fp8, marlin, moe_int4, ops  # noqa: E402

GROUP = 128
EPS = 1e-6
DECODE_ROWS = 16  # most rows of a captured decode step


# ------------------------------------------------------------------- the cases
def listed():
    # Qwen3-8B: hidden 4096, 32 query and 8 key/value heads of 128, MLP 12288
    dense = {"kind": "layer", "hidden": 4096, "q_dim": 4096, "kv_dim": 1024, "inter": 12288}
    # DeepSeek-V2-Lite's dense layer, one fp32 scale per 128x128 block
    block = {"kind": "fp8", "hidden": 2048, "inter": 10944}
    # Qwen1.5-MoE-A2.7B: 60 experts of 1408, top 4, a shared expert of 5632
    qwen15 = {"kind": "moe", "hidden": 2048, "inter": 1408, "experts": 60, "top_k": 4, "shared": 5632,
              "norm": False}
    # Qwen3-30B-A3B: 128 experts of 768, top 8 with renormalised weights
    qwen3 = {"kind": "moe", "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8, "shared": 0,
             "norm": True}
    return [
        # one projection of a small model, called eagerly for one token
        {"name": "int4_call_m1", "kind": "call", "rows": 1, "out": 3072, "in": 1024},
        # single-stream decode, one layer of the captured chain
        {"name": "int4_layer_m1", **dense, "rows": 1},
        # a small decode batch (odd), one layer of the captured chain
        {"name": "int4_layer_m13", **dense, "rows": 13},
        # a server's decode batch, or the rows of speculative decoding
        {"name": "int4_layer_m48", **dense, "rows": 48},
        # a short prompt, its length no multiple of a tile
        {"name": "int4_layer_m500", **dense, "rows": 500},
        # a long prompt, or one chunk of a very long one
        {"name": "int4_layer_m4096", **dense, "rows": 4096},
        # decode batch on FP8 weights, four layers in one graph
        {"name": "fp8_linears_m8", **block, "rows": 8, "layers": 4, "bf16": True},
        # prompt on FP8 weights
        {"name": "fp8_linears_m2000", **block, "rows": 2000, "layers": 1, "bf16": True},
        # single-stream MoE decode, four layers in one graph
        {"name": "moe_int4_t1", **qwen15, "rows": 1, "layers": 4, "format": "int4"},
        # batched MoE decode
        {"name": "moe_int4_t16", **qwen15, "rows": 16, "layers": 2, "format": "int4"},
        # MoE prefill with many small experts
        {"name": "moe_int4_t512", **qwen3, "rows": 512, "layers": 1, "format": "int4"},
        # MoE prefill on FP8 experts, with a shared expert
        {"name": "moe_fp8_t1000", **qwen15, "rows": 1000, "layers": 1, "format": "fp8"},
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("call", "layer", "layer", "fp8", "moe", "moe"))
    if kind == "call":
        return {"kind": kind, "rows": _spread(rng, 1, DECODE_ROWS), "out": 64 * _spread(rng, 16, 384),
                "in": 128 * _spread(rng, 8, 32)}
    if kind == "layer":
        return {"kind": kind, "rows": _spread(rng, 1, 4096), "hidden": 128 * rng.randint(8, 32),
                "q_dim": 128 * rng.randint(8, 32), "kv_dim": 64 * rng.randint(2, 16),
                "inter": 128 * rng.randint(20, 96)}
    if kind == "fp8":
        rows = _spread(rng, 1, 2000)
        return {"kind": kind, "rows": rows, "hidden": 64 * rng.randint(16, 40),
                "inter": 64 * rng.randint(32, 171), "layers": 4 if rows <= DECODE_ROWS else 1,
                "bf16": rng.random() < 0.75}
    experts = rng.choice((60, 64, 128))
    top_k = rng.choice((4, 6, 8))
    rows = _spread(rng, 1, min(1000, 4096 // top_k, 32 * (4096 // experts)))
    inter = 128 * rng.randint(6, 11)
    return {"kind": kind, "rows": rows, "hidden": 256 * rng.randint(4, 8), "inter": inter,
            "experts": experts, "top_k": top_k, "shared": rng.choice((0, inter, 2 * inter, 4 * inter)),
            "norm": rng.random() < 0.5, "layers": 2 if rows <= DECODE_ROWS else 1,
            "format": rng.choice(("int4", "int4", "fp8"))}


# --------------------------------------------------------- inputs from the seed
class _Source:
    """Tensors made from the seed alone: the i-th one asked for is always the same."""

    def __init__(self, seed):
        self.seed, self.asked = int(seed), 0
        self.gen = torch.Generator(device="cuda")

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        self.asked += 1
        self.gen.manual_seed(self.seed * 1009 + self.asked)
        return (torch.randn(shape, generator=self.gen, device="cuda") * std).to(dtype)


def _int4(src, *shape):
    """A weight (..., out, in) ~ N(0, 0.02), rounded to 4 bits with one fp16 scale and one whole
    zero point per 128 inputs: codes u8, scales fp16 and zeros fp16 (..., out, in / 128)."""
    w = src.normal(*shape, std=0.02).unflatten(-1, (-1, GROUP))
    lo, hi = w.amin(-1), w.amax(-1)
    scale = ((hi - lo) / 15).clamp_min(1e-8).half()
    zero = torch.round(-lo / scale.float()).clamp_(0, 15)
    q = torch.round(w / scale.float()[..., None]).add_(zero[..., None]).clamp_(0, 15)
    return q.to(torch.uint8).flatten(-2), scale, zero.half()


def _int4_value(q, scale, zero):
    w = (q.unflatten(-1, (-1, GROUP)).double() - zero.double()[..., None]) * scale.double()[..., None]
    return w.flatten(-2)


def _fp8(src, *shape):
    """A weight (..., out, in) ~ N(0, 0.02) in e4m3 with one scale per 128x128 block: codes
    (float8_e4m3fn) and scales fp32.  The scales have few bits and every block holds the largest
    code, so that quantizing the values again gives these codes and scales."""
    rows, cols = shape[-2:]
    w = src.normal(*shape, std=0.02)
    w = torch.nn.functional.pad(w, (0, -cols % 128, 0, -rows % 128))
    w = w.unflatten(-1, (-1, 128)).unflatten(-3, (-1, 128))
    scale = (w.abs().amax((-3, -1)) / 448).bfloat16().float()
    v = (w / scale[..., :, None, :, None]).clamp_(-448, 448)
    v[..., 0, :, 0] = 448
    q = v.to(torch.float8_e4m3fn).flatten(-4, -3).flatten(-2)
    return q[..., :rows, :cols].contiguous(), scale


def _fp8_value(q, scale, dtype=torch.float64):
    rows, cols = q.shape[-2:]
    s = scale.to(dtype).repeat_interleave(128, -2)[..., :rows, :]
    return q.to(dtype) * s.repeat_interleave(128, -1)[..., :cols]


def _layer_inputs(case, seed):
    src, M, h = _Source(seed), case["rows"], case["hidden"]
    n_qkv = case["q_dim"] + 2 * case["kv_dim"]
    return {
        "x": src.normal(M, h),
        "delta": src.normal(M, h, std=0.5, dtype=torch.float16),
        "ctx": src.normal(M, case["q_dim"], dtype=torch.float16),  # what attention returns
        "ln1": (1 + src.normal(h, std=0.1)).half(),
        "ln2": (1 + src.normal(h, std=0.1)).half(),
        "qkv": _int4(src, n_qkv, h),
        "o": _int4(src, h, case["q_dim"]),
        "gate_up": _int4(src, 2 * case["inter"], h),
        "down": _int4(src, h, case["inter"]),
    }


def _call_inputs(case, seed):
    src = _Source(seed)
    return {"a": src.normal(case["rows"], case["in"], dtype=torch.float16),
            "w": _int4(src, case["out"], case["in"])}


def _fp8_shapes(case):
    h, i = case["hidden"], case["inter"]
    return ((h, h), (i, h), (h, i))


def _fp8_inputs(case, seed):
    src = _Source(seed)
    dtype = torch.bfloat16 if case["bf16"] else torch.float16
    return [(src.normal(case["rows"], k, dtype=dtype), *_fp8(src, n, k))
            for _ in range(case["layers"]) for n, k in _fp8_shapes(case)]


def _moe_inputs(case, seed):
    """One layer after another: activations, router weights, routed and shared projections."""
    src, h = _Source(seed), case["hidden"]
    weight = _int4 if case["format"] == "int4" else _fp8
    for _ in range(case["layers"]):
        one = {"x": src.normal(case["rows"], h),
               "gate_w": src.normal(case["experts"], h, std=h ** -0.5, dtype=torch.float16),
               "shared_gate_w": src.normal(h, std=h ** -0.5, dtype=torch.float16)}
        for name, experts, inter in (("routed", case["experts"], case["inter"]),
                                     ("shared", 1, case["shared"])):
            one[name] = None if not inter else {
                proj: weight(src, experts, *shape)
                for proj, shape in (("gate", (inter, h)), ("up", (inter, h)), ("down", (h, inter)))}
        yield one


# ------------------------------------------------------------------ what a program keeps
def _marlin(w):
    q, scale, zero = w
    std = marlin.pack_gptq_qweight(q.to(torch.int32), xp=torch)
    scales, zeros = marlin.build_marlin_scales_zeros(scale.float(), zero.to(torch.int32), GROUP, xp=torch)
    return {"qweight": marlin.marlin_repack(std, q.shape[1], q.shape[0]), "scales": scales, "zeros": zeros}


def _stack(weights, fmt):
    out = {"group": GROUP, "layout": "tile16x128"}
    if fmt != "int4":
        out["format"] = fmt
    for proj, w in weights.items():
        if fmt == "int4":
            q, scale, zero = w
            out.update(moe_int4.stack_tiles(proj, q[..., ::2] | (q[..., 1::2] << 4), scale, zero, GROUP))
        else:
            out.update(moe_int4.stack_lowp(fmt, proj, _fp8_value(*w, dtype=torch.float32)))
    return out


def _captured(step):
    """`step(stream)`, warmed up and captured in a graph, as a decode loop keeps it."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step(stream)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        step(stream)
    return graph


def _prepare_call(case, seed):
    d = _call_inputs(case, seed)
    return {"a": d["a"], "w": _marlin(d["w"]), "ws": marlin.make_workspace(case["out"]),
            "out": torch.empty(case["rows"], case["out"], dtype=torch.float16, device="cuda")}


def _run_call(s):
    w = s["w"]
    return marlin.gemm_fast(s["a"], w["qweight"], w["scales"], w["zeros"], s["out"].shape[1], s["a"].shape[1],
                            stream=torch.cuda.current_stream(), workspace=s["ws"], out=s["out"])


def _prepare_layer(case, seed):
    d, M, h = _layer_inputs(case, seed), case["rows"], case["hidden"]
    weights = {k: _marlin(d[k]) if isinstance(d[k], tuple) else d[k]
               for k in ("ln1", "ln2", "qkv", "o", "gate_up", "down")}
    if M <= DECODE_ROWS:
        g = DecodeLayerGraph(weights, M, h, case["q_dim"], case["inter"], eps=EPS)
        g.x.copy_(d["x"])
        g.pending.copy_(d["delta"])
        return {"graph": g.capture()}

    def buf(n, dtype=torch.float16):
        return torch.empty(M, n, dtype=dtype, device="cuda")

    n = {k: weights[k]["scales"].shape[1] for k in ("qkv", "o", "gate_up", "down")}
    return {"w": weights, "n": n, "inter": case["inter"], "x": d["x"], "delta": d["delta"], "ctx": d["ctx"],
            "ws": {k: marlin.make_workspace(v) for k, v in n.items()},
            "norm1": (buf(h, torch.float32), buf(h)), "norm2": (buf(h, torch.float32), buf(h)),
            "act": buf(case["inter"]), **{"out_" + k: buf(v) for k, v in n.items()}}


def _run_layer(s):
    if "graph" in s:
        g = s["graph"]
        g.replay()
        return {"qkv": g.qkv, "x": g.x_out, "delta": g.pending_out}
    stream = torch.cuda.current_stream()

    def linear(name, a):
        p = s["w"][name]
        return marlin.gemm_fast(a, p["qweight"], p["scales"], p["zeros"], s["n"][name], a.shape[1], stream=stream,
                                workspace=s["ws"][name], out=s["out_" + name])

    x, h = ops.add_rmsnorm(s["x"], s["delta"], s["w"]["ln1"], EPS, out=s["norm1"], stream=stream)
    qkv = linear("qkv", h)
    o = linear("o", s["ctx"])
    x, h = ops.add_rmsnorm(x, o, s["w"]["ln2"], EPS, out=s["norm2"], stream=stream)
    gate_up = linear("gate_up", h)
    inter = s["inter"]
    act = ops.swiglu(gate_up[:, :inter], gate_up[:, inter:], out=s["act"], stream=stream)
    return {"qkv": qkv, "x": x, "delta": linear("down", act)}


def _prepare_fp8(case, seed):
    calls = [{"x": x, "q": q.view(torch.uint8), "scale": scale,
              "out": torch.empty(x.shape[0], q.shape[0], dtype=x.dtype, device="cuda")}
             for x, q, scale in _fp8_inputs(case, seed)]
    state = {"calls": calls}
    if case["rows"] <= DECODE_ROWS:
        state["graph"] = _captured(lambda stream: _fp8_step(calls, stream))
    return state


def _fp8_step(calls, stream):
    for c in calls:
        fp8.fp8_gemv_block(c["x"], c["q"], c["scale"], out=c["out"], stream=stream)


def _run_fp8(s):
    if "graph" in s:
        s["graph"].replay()
    else:
        _fp8_step(s["calls"], torch.cuda.current_stream())
    return [c["out"] for c in s["calls"]]


def _prepare_moe(case, seed):
    T, h, layers = case["rows"], case["hidden"], []
    for d in _moe_inputs(case, seed):
        bufs = {"logits": torch.empty(T, case["experts"], device="cuda"), "slogit": torch.empty(T, device="cuda")}
        shared = d["shared"] and _stack(d["shared"], case["format"])
        layers.append({"x": d["x"], "gate_w": d["gate_w"], "stacked": _stack(d["routed"], case["format"]),
                       "top_k": case["top_k"],
                       "kw": {"E": case["experts"], "hidden": h, "inter": case["inter"], "norm": case["norm"],
                              "shared": shared, "shared_inter": case["shared"],
                              "shared_gate_w": d["shared_gate_w"] if shared else None, "bufs": bufs}})
    state = {"layers": layers}
    if T <= DECODE_ROWS:
        state["graph"] = _captured(lambda stream: _moe_step(layers, stream))
    return state


def _moe_step(layers, stream):
    for d in layers:
        moe_int4.moe_branch(d["x"], d["gate_w"], d["stacked"], d["top_k"], stream=stream, **d["kw"])


def _run_moe(s):
    if "graph" in s:
        s["graph"].replay()
    else:
        _moe_step(s["layers"], torch.cuda.current_stream())
    bufs = [d["kw"]["bufs"] for d in s["layers"]]
    return {"y": [b["out"] for b in bufs], "logits": [b["logits"] for b in bufs],
            "weights": [b["topk_w"] for b in bufs], "experts": [b["topk_ids"] for b in bufs]}


_PREPARE = {"call": _prepare_call, "layer": _prepare_layer, "fp8": _prepare_fp8, "moe": _prepare_moe}
_RUN = {"call": _run_call, "layer": _run_layer, "fp8": _run_fp8, "moe": _run_moe}


def prepare(case, seed):
    return {"kind": case["kind"], **_PREPARE[case["kind"]](case, seed)}


def run(state):
    return _RUN[state["kind"]](state)


# ----------------------------------------------------------- what a pass cannot do without
def work(case):
    M = case["rows"]
    nbytes = flops = 0.0

    def int4(n, k):  # codes, fp16 scales, packed 4-bit zeros
        return n * k / 2 + n * (k / GROUP) * 2.5

    def block(n, k):
        return n * k + 4 * math.ceil(n / 128) * math.ceil(k / 128)

    if case["kind"] == "call":
        n, k = case["out"], case["in"]
        nbytes, flops = int4(n, k) + 2 * M * (n + k), 2.0 * M * n * k
    elif case["kind"] == "layer":
        h, q, i = case["hidden"], case["q_dim"], case["inter"]
        for n, k in ((q + 2 * case["kv_dim"], h), (h, q), (2 * i, h), (h, i)):
            nbytes += int4(n, k)
            flops += 2.0 * M * n * k
        # x and the branch in, x, the branch and qkv out; above the decode graph ctx in
        nbytes += M * (h * 12 + 2 * (q + 2 * case["kv_dim"]) + (2 * q if M > DECODE_ROWS else 0))
    elif case["kind"] == "fp8":
        for n, k in _fp8_shapes(case):
            nbytes += case["layers"] * (block(n, k) + 2 * M * (n + k))
            flops += case["layers"] * 2.0 * M * n * k
    else:
        h, E, k = case["hidden"], case["experts"], case["top_k"]
        size = int4 if case["format"] == "int4" else block
        reached = E * (1 - (1 - k / E) ** M)  # experts that some token goes to, on average
        for experts, each, inter in ((reached, k, case["inter"]), (1, 1, case["shared"])):
            if inter:
                nbytes += experts * (2 * size(inter, h) + size(h, inter))
                flops += 6.0 * M * each * h * inter
        nbytes += 2 * E * h + 8.0 * M * h
        flops += 2.0 * M * E * h
        nbytes, flops = nbytes * case["layers"], flops * case["layers"]
    return {"bytes": nbytes, "flops": flops}


# --------------------------------------------------------------------- right answers
def tolerance(case):
    # About four times what the outputs were off their 64-bit values by: one
    # rounding of the result to 16 bits for a call and the FP8 linears (2.1e-4,
    # bf16 1.7e-3), several in a row in a layer (7.1e-4) and a MoE layer (4.8e-4;
    # there a token whose last chosen expert ties with the next one may differ).
    return {"call": {"rel": 1e-3}, "layer": {"rel": 3e-3},
            "fp8": {"rel": 7e-3} if case.get("bf16") else {"rel": 1.2e-3},
            "moe": {"rel": 2e-3, "max": 0.4, "differ": 1e-3}}[case["kind"]]


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_layer(case, seed):
    d = _layer_inputs(case, seed)

    def linear(name, a):
        return a @ _int4_value(*d[name]).T

    x = d["x"].double() + d["delta"].double()
    qkv = linear("qkv", _norm(x, d["ln1"]))
    ctx = qkv[:, :case["q_dim"]] if case["rows"] <= DECODE_ROWS else d["ctx"].double()
    x = x + linear("o", ctx)
    gate, up = linear("gate_up", _norm(x, d["ln2"])).chunk(2, -1)
    return {"qkv": qkv, "x": x, "delta": linear("down", _silu(gate) * up)}


def _exact_moe(case, seed):
    value = _int4_value if case["format"] == "int4" else _fp8_value
    out = {"y": [], "logits": [], "weights": [], "experts": []}
    for d in _moe_inputs(case, seed):
        x = d["x"].double()
        logits = x @ d["gate_w"].double().T
        w, ids = torch.softmax(logits, -1).topk(case["top_k"], -1)
        if case["norm"]:
            w = w / w.sum(-1, keepdim=True)
        y = torch.zeros_like(x)

        def expert(weights, e, rows):
            g, u, dn = (value(*(v[e] for v in weights[p])) for p in ("gate", "up", "down"))
            return (_silu(rows @ g.T) * (rows @ u.T)) @ dn.T

        for e in ids.unique().tolist():
            t, slot = (ids == e).nonzero(as_tuple=True)
            y.index_add_(0, t, expert(d["routed"], e, x[t]) * w[t, slot, None])
        if d["shared"]:
            y += expert(d["shared"], 0, x) * torch.sigmoid(x @ d["shared_gate_w"].double())[:, None]
        out["y"].append(y)
        out["logits"].append(logits)
        out["weights"].append(w)
        out["experts"].append(None)
    return out


def exact(case, seed):
    if case["kind"] == "call":
        d = _call_inputs(case, seed)
        return d["a"].double() @ _int4_value(*d["w"]).T
    if case["kind"] == "fp8":
        return [x.double() @ _fp8_value(q, scale).T for x, q, scale in _fp8_inputs(case, seed)]
    return _exact_layer(case, seed) if case["kind"] == "layer" else _exact_moe(case, seed)

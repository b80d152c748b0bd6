"""The work a decode engine hands to this library, as cases that can be timed and compared.

A case is one pass through the public entry points, as the engine makes it:

- ``linear``: the projections of a few layers, one call each. Up to 8 rows go to lx_gemv_w, more to lx_gemm_w.
- ``experts``: the routed experts of a few layers, one lx_moe_route (lx_router_route where the router's shape allows
  it) and one experts call each. Up to 8 tokens go to lx_moe_experts_decode, more to lx_moe_experts_grouped.

A pass of at most 64 rows is a decode step: it is captured once into a graph through lx_rt_capture_* and replayed, on a
stream made by lx_rt_stream_create, which is how the engine runs its decode steps. More rows are a prefill: its calls
are issued one by one on the same stream. The layers have weights of their own, and a decode state holds
enough of them that no pass finds its weights in the 256 MB Infinity Cache (a model's layers do not fit it either).

Weights are N(0, 0.02) bf16 masters quantised by the library's own quantiser, activations N(0, 1) bf16, router logits
N(0, 1): the distributions the configurations state.
"""

import ctypes
import math
import os

import torch

from dromos_amd import abi
from dromos_amd.formats import Weight, alloc_quantized

MATHS = {"bf16": abi.MATH_BF16, "int8": abi.MATH_INT8, "fp8": abi.MATH_FP8, "fp4": abi.MATH_FP4}
NATIVE_MATH = {"bf16": "bf16", "int8": "int8", "fp8": "fp8", "nvfp4": "fp4"}
BYTES_PER_VALUE = {"bf16": 2.0, "int8": 1.0, "fp8": 1.0, "nvfp4": 0.5625}  # nvfp4: with its block scales
DECODE_ROWS = 64           # up to here a pass is a decode step (a graph)
COLD_BYTES = 400 << 20     # what a decode state's weights come to at least
MAX_LAYERS = 24


def linear(name, fmt, rows, n, k, layers, math="bf16", invariant=False, y="f32"):
    return {"name": name, "kind": "linear", "format": fmt, "math": math, "rows": rows, "n": n, "k": k, "layers": layers,
            "invariant": invariant, "y": y}


def experts(name, fmt, tokens, n_experts, top_k, latent, inter, layers, math="bf16"):
    return {"name": name, "kind": "experts", "format": fmt, "math": math, "tokens": tokens, "experts": n_experts, "top_k": top_k,
            "latent": latent, "inter": inter, "layers": layers}


def listed():
    return [
        # One stream decoding: a layer's widest INT8 projection (the benchmark's headline shape).
        linear("linear_int8_14336x4096_m1", "int8", 1, 14336, 4096, 8),
        # One stream decoding: a square BF16 projection, the smallest of the dense single-row products.
        linear("linear_bf16_4096x4096_m1", "bf16", 1, 4096, 4096, 13),
        # One stream decoding: NVFP4 on long rows (a down projection).
        linear("linear_nvfp4_4096x14336_m1", "nvfp4", 1, 4096, 14336, 14),
        # A few drafted tokens verified together, on the width of a model whose rows are not a power of two.
        linear("linear_fp8_11008x4096_m4", "fp8", 4, 11008, 4096, 10),
        # 32 streams: the QKV projection of the FP8 decode layer.
        linear("linear_fp8_6144x4096_m32", "fp8", 32, 6144, 4096, 18),
        # 64 streams in the batch-invariant mode on an NVFP4 weight.
        linear("linear_nvfp4_14336x4096_m64", "nvfp4", 64, 14336, 4096, 14, invariant=True),
        # A prompt: 4096 tokens through an FP8 projection, BF16 outputs for the next operator.
        linear("linear_fp8_14336x4096_m4096", "fp8", 4096, 14336, 4096, 1, y="bf16"),
        # The ragged end of a prompt under the INT8 math: activations quantised inside the call, rows that are not a power of two.
        linear("linear_int8_4096x11008_m515_int8", "int8", 515, 4096, 11008, 2, math="int8"),
        # One stream decoding through routed experts: eight of 64 BF16 experts.
        experts("experts_bf16_e64_t1", "bf16", 1, 64, 8, 2048, 1024, 4),
        # 32 streams through the FP8 decode layer's 128 experts.
        experts("experts_fp8_e128_t32", "fp8", 32, 128, 8, 4096, 1536, 1),
        # A prompt of 2048 tokens through NVFP4 experts (the published recipe holds the experts in NVFP4).
        experts("experts_nvfp4_e128_t2048", "nvfp4", 2048, 128, 8, 4096, 1536, 1),
        # A small model's single token: router, four of 64 INT8 experts. The launches and their gaps weigh most here.
        experts("experts_int8_e64_t1_small", "int8", 1, 64, 4, 1024, 512, 4),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: rows from 1 to 4096 (tokens to 2048), every format, the native maths on more than 8 rows, N and K
    over the range the listed shapes span, some of them odd."""
    fmt = rng.choice(["bf16", "int8", "fp8", "nvfp4"])
    if rng.random() < 0.6:
        rows = _log_int(rng, 1, 4096)
        while True:
            n, k = _log_int(rng, 1024, 16384), _log_int(rng, 1024, 14336)
            n = n if rng.random() < 0.2 else (n + 15) // 16 * 16
            k = (k + 31) // 32 * 32 if rng.random() < 0.3 else (k + 255) // 256 * 256
            if 2.0 * rows * n * k <= 4.8e11 and n * k <= 14336 * 8192:
                break
        quantised = rows > 8 and fmt != "bf16" and rng.random() < 0.25
        per_layer = n * k * BYTES_PER_VALUE[fmt]
        layers = max(1, min(MAX_LAYERS, math.ceil(COLD_BYTES / per_layer))) if rows <= DECODE_ROWS else 1
        case = linear("", fmt, rows, n, k, layers, NATIVE_MATH[fmt] if quantised else "bf16", rows <= DECODE_ROWS and rng.random() < 0.25,
                      rng.choice(["f32", "bf16"]))
    else:
        while True:
            tokens = _log_int(rng, 1, 2048)
            n_experts, top_k = rng.choice([16, 32, 64, 96, 128]), rng.choice([2, 4, 6, 8])
            latent = (_log_int(rng, 1024, 4096) + 63) // 64 * 64
            inter = (_log_int(rng, 512, 2048) + 31) // 32 * 32
            if 6.0 * tokens * top_k * latent * inter <= 4.8e11 and 3.0 * n_experts * latent * inter * BYTES_PER_VALUE[fmt] <= 2.2e9:
                break
        quantised = tokens > 8 and fmt != "bf16" and rng.random() < 0.2
        per_layer = 3.0 * n_experts * latent * inter * BYTES_PER_VALUE[fmt]
        layers = max(1, min(4, math.ceil(COLD_BYTES / per_layer))) if tokens <= DECODE_ROWS else 1
        case = experts("", fmt, tokens, n_experts, top_k, latent, inter, layers, NATIVE_MATH[fmt] if quantised else "bf16")
    del case["name"]
    return case


# ---- what a program keeps: the library, its stream, the weights, the buffers, the captured decode step ------------


_program = {}


def _library():
    if not _program:
        lx = abi.load_hip()
        stream = ctypes.c_void_p()
        assert lx.lib.lx_rt_stream_create(ctypes.byref(stream)) == 0
        _program.update(lx=lx, stream=stream.value)
    return _program["lx"], _program["stream"]


def _quantised(lx, fmt, lead, n, k, generator):
    """A weight [n, k] or stack [E, n, k] in `fmt`, from N(0, 0.02) bf16 values."""
    rows = n * (lead or 1)
    master = torch.randn(rows, k, generator=generator, device="cuda", dtype=torch.bfloat16).mul_(0.02)
    if fmt == "bf16":
        return Weight(abi.W_BF16, master)
    out = alloc_quantized(abi.FORMATS[fmt], rows, k, "cuda")
    struct = out.lx()
    assert lx.status("quantize_weight", master, ctypes.pointer(struct), rows, k) == 0
    out.glob = float(struct.global_)
    return out


class State:
    """Inputs, weights and buffers of one pass, and its calls: [(entry point, arguments)], or the graph that holds them."""

    def __init__(self, lx, stream):
        self.lx, self.stream = lx, stream
        self.keep, self.calls, self.outputs = [], [], []
        self.graph = None

    def add(self, name, *args):
        self.calls.append((name, tuple(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args) + (self.stream,)))
        self.keep += args

    def issue(self):
        for name, args in self.calls:
            status = self.lx.status(name, *args)
            if status != 0:
                raise RuntimeError(f"lx_{name} returned {status}")

    def capture(self):
        lib, graph = self.lx.lib, ctypes.c_void_p()
        assert lib.lx_rt_capture_begin(self.stream) == 0
        self.issue()
        assert lib.lx_rt_capture_end(self.stream, ctypes.byref(graph)) == 0
        self.graph = graph

    def __del__(self):
        if self.graph is not None:
            self.lx.lib.lx_rt_graph_destroy(self.graph)


def _linear_state(case, lx, stream, g):
    s = State(lx, stream)
    fmt, rows, n, k = case["format"], case["rows"], case["n"], case["k"]
    mathid, y_type = MATHS[case["math"]], {"f32": torch.float32, "bf16": torch.bfloat16}[case["y"]]
    workspace = torch.empty(max(256, int(lx.size("gemm_workspace_bytes", rows, k, mathid))), dtype=torch.uint8, device="cuda")
    for _ in range(case["layers"]):
        w = _quantised(lx, fmt, None, n, k, g)
        struct = w.lx()
        x = torch.randn(rows, k, generator=g, device="cuda", dtype=torch.bfloat16)
        y = torch.empty(rows, n, dtype=y_type, device="cuda")
        s.keep += [w, struct]
        operands = (x, abi.BF16, k, ctypes.pointer(struct))
        tail = (None, abi.F32, y, abi.DTYPE[y_type], n, rows, n, k, 1.0, 0.0)
        if rows <= 8:
            s.add("gemv_w", *operands, *tail)
        else:
            s.add("gemm_w", *operands, mathid, *tail, workspace)
        s.outputs.append(y)
    return s


def _experts_state(case, lx, stream, g):
    s = State(lx, stream)
    fmt, t, e, top_k, latent, inter = (case[key] for key in ("format", "tokens", "experts", "top_k", "latent", "inter"))
    mathid = MATHS[case["math"]]
    few = t <= 8
    nbytes = lx.size("moe_decode_workspace_bytes", t, inter, top_k) if few else lx.size("moe_grouped_workspace_bytes", t, latent, inter, e, top_k, mathid)
    workspace = torch.empty(max(256, int(nbytes)), dtype=torch.uint8, device="cuda")
    for _ in range(case["layers"]):
        gate_up, down = _quantised(lx, fmt, e, 2 * inter, latent, g), _quantised(lx, fmt, e, latent, inter, g)
        structs = gate_up.lx(), down.lx()
        s.keep += [gate_up, down, structs]
        x = torch.randn(t, latent, generator=g, device="cuda", dtype=torch.bfloat16)
        ids = torch.empty(t, top_k, dtype=torch.int32, device="cuda")
        weights = torch.empty(t, top_k, dtype=torch.float32, device="cuda")
        entropy, confidence = torch.empty(t, device="cuda"), torch.empty(t, device="cuda")
        out = torch.empty(t, latent, dtype=torch.float32, device="cuda")
        if few and latent <= 2048:  # what lx_router_route takes: the router's product and the routing in one call
            router = torch.randn(e, latent, generator=g, device="cuda").mul_(latent**-0.5)
            logits, ticket = torch.empty(t, e, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
            s.add("router_route", x.float(), latent, router, None, logits, None, ids, weights, entropy, confidence, ticket, t, e, latent, top_k)
        else:
            logits = torch.randn(t, e, generator=g, device="cuda")
            s.add("moe_route", logits, None, ids, weights, entropy, confidence, t, e, top_k)
        pair = ctypes.pointer(structs[0]), ctypes.pointer(structs[1])
        if few:
            s.add("moe_experts_decode", x, ids, weights, *pair, out, workspace, t, latent, inter, top_k)
        else:
            s.add("moe_experts_grouped", x, ids, weights, *pair, mathid, out, workspace, t, latent, inter, e, top_k)
        s.outputs += [ids, weights, entropy, confidence, out]
    return s


def prepare(case, seed):
    lx, stream = _library()
    g = torch.Generator(device="cuda").manual_seed(seed)
    make = _linear_state if case["kind"] == "linear" else _experts_state
    state = make(case, lx, stream, g)
    torch.cuda.synchronize()
    if (case["rows"] if case["kind"] == "linear" else case["tokens"]) <= DECODE_ROWS:
        # The mode is read when a call is made: a captured step keeps the one it was captured in.
        if case.get("invariant"):
            os.environ["LX_BATCH_INVARIANT"] = "1"
        try:
            state.capture()
        finally:
            os.environ.pop("LX_BATCH_INVARIANT", None)
    return state


def run(state):
    if state.graph is not None:
        status = state.lx.lib.lx_rt_graph_launch(state.graph, state.stream)
        if status != 0:
            raise RuntimeError(f"lx_rt_graph_launch returned {status}")
    else:
        state.issue()
    return state.outputs


def work(case):
    """Weights read once (of the experts, those the tokens are expected to pick), activations read once, outputs written
    once; two operations per weight value and row."""
    per_value = BYTES_PER_VALUE[case["format"]]
    if case["kind"] == "linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        nbytes = n * k * per_value + rows * k * 2 + rows * n * (4 if case["y"] == "f32" else 2)
        flops = 2.0 * rows * n * k
    else:
        t, e, top_k, latent, inter = (case[key] for key in ("tokens", "experts", "top_k", "latent", "inter"))
        picked = e * (1.0 - (1.0 - top_k / e) ** t)
        nbytes = picked * 3 * latent * inter * per_value + t * latent * 6 + t * e * 4
        flops = 6.0 * t * top_k * latent * inter
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    """Measured against the same products in 64 bits, times about four. The f32 sums: 0.7 to 1.0e-7 in norm, 7e-7 at most
    (rows of 4096 and 14336 values). BF16 outputs are those sums rounded once: where two sums fall on either side of a
    tie they differ by one unit, 2^-7 of the value at most, one value in some ten thousand. The experts' BF16
    intermediate rows do the same one stage earlier: 2.2e-5 and 1.4e-3 at 2048 tokens with exact sums. Under a quantised
    math such a value of an intermediate row moves by a whole 8- or 4-bit step."""
    if case["kind"] == "experts":
        return {"rel": 1e-4, "max": 6e-3} if case["math"] == "bf16" else {"rel": 1e-3, "max": 1e-1}
    return {"rel": 2e-4, "max": 8e-3} if case["y"] == "bf16" else {"rel": 5e-7, "max": 4e-6}


# ---- the same outputs in 64 bits, without the library ---------------------------------------------------------------


def _e2m1(v):
    """The nearest e2m1 value (ties to the even code), saturating at 6."""
    grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device=v.device)
    low, high = torch.tensor([0.25, 1.25, 2.5, 5.0], device=v.device), torch.tensor([0.75, 1.75, 3.5], device=v.device)
    a = v.abs()
    code = sum((a > t).int() for t in low) + sum((a >= t).int() for t in high)
    return torch.copysign(grid[code.long()], v)


def _e4m3(v):
    return v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).float()


def _divided(a, b):
    """a / b in f32 as IEEE rounds it (a double holds the quotient closely enough for one rounding)."""
    return (a.double() / b.double()).float()


def _weight_values(master, fmt, top=None):
    """What the stored rows stand for, before the row factor (f32, exact), and the row factor [rows, 1] (f64). `top` is
    the largest magnitude of the whole matrix or stack that the rows are part of (NVFP4 has one global factor)."""
    w = master.float()
    if fmt == "bf16":
        return w, torch.ones(w.shape[0], 1, device=w.device, dtype=torch.float64)
    if fmt == "nvfp4":
        scale = _divided(w.abs().max() if top is None else top, torch.tensor(2688.0, device=w.device))
        blocks = w.view(w.shape[0], -1, 16)
        s = _e4m3(_divided(blocks.abs().amax(2), 6.0 * scale))
        step = (s * scale).unsqueeze(2)
        codes = torch.where(step > 0, _e2m1(_divided(blocks, step)), torch.zeros_like(blocks))
        return (codes * s.unsqueeze(2)).view_as(w), scale.double().expand(w.shape[0], 1)
    s = _divided(w.abs().amax(1, keepdim=True), torch.tensor(127.0 if fmt == "int8" else 448.0, device=w.device))
    v = _divided(w, s)
    return (v.round().clamp(-127.0, 127.0) if fmt == "int8" else _e4m3(v)), s.double()


def _activation_values(x, math_name):
    """The same of bf16 activation rows under a math: quantised per row, by a reciprocal (f32)."""
    x = x.float()
    if math_name == "bf16":
        return x, torch.ones(x.shape[0], 1, device=x.device, dtype=torch.float64)
    a = x.abs().amax(1, keepdim=True)
    if math_name == "fp4":
        g = _divided(a, torch.full_like(a, 2688.0))
        blocks = x.view(x.shape[0], -1, 16)
        s = _e4m3(_divided(blocks.abs().amax(2), 6.0 * g))
        step = (s * g).unsqueeze(2)
        codes = torch.where(step > 0, _e2m1(blocks * _divided(torch.ones_like(step), step)), torch.zeros_like(blocks))
        return (codes * s.unsqueeze(2)).view_as(x), g.double()
    top = torch.full_like(a, 127.0 if math_name == "int8" else 448.0)
    v = x * _divided(top, a)
    return (v.round().clamp(-127.0, 127.0) if math_name == "int8" else _e4m3(v)), _divided(a, top).double()


def _product(x, master, fmt, math_name, top=None):
    values, factor = _weight_values(master, fmt, top)
    rows, scale = _activation_values(x, math_name)
    return (rows.double() @ values.double().t().contiguous()) * scale * factor.t()


def _routing(logits, top_k):
    """Ids (in the order of the scores), weights, entropy and confidence of every token."""
    logits = logits.double()
    picked, ids = logits.topk(top_k, dim=1)
    p = torch.softmax(logits, 1)
    return ids, torch.softmax(picked, 1), -(p * p.clamp_min(1e-9).log()).sum(1), p.amax(1)


def exact(case, seed):
    """What run() returns, computed in 64 bits from the same inputs (ids, which are whole numbers, have None). The
    quantised values themselves are the formats' own and taken as given, and so are the experts' bf16 intermediate rows."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)

    outputs, fmt, math_name = [], case["format"], case["math"]
    for _ in range(case["layers"]):
        if case["kind"] == "linear":
            master = normal(case["n"], case["k"], dtype=torch.bfloat16).mul_(0.02)
            outputs.append(_product(normal(case["rows"], case["k"], dtype=torch.bfloat16), master, fmt, math_name))
            continue
        t, e, top_k, latent, inter = (case[key] for key in ("tokens", "experts", "top_k", "latent", "inter"))
        gate_up = normal(e * 2 * inter, latent, dtype=torch.bfloat16).mul_(0.02)
        down = normal(e * latent, inter, dtype=torch.bfloat16).mul_(0.02)
        x = normal(t, latent, dtype=torch.bfloat16)
        if t <= 8 and latent <= 2048:
            logits = x.double() @ normal(e, latent).mul_(latent**-0.5).double().t().contiguous()
        else:
            logits = normal(t, e)
        ids, weights, entropy, confidence = _routing(logits, top_k)
        out = torch.zeros(t, latent, dtype=torch.float64, device="cuda")
        tops = [m.float().abs().max() if fmt == "nvfp4" else None for m in (gate_up, down)]
        for expert in range(e):
            token, slot = (ids == expert).nonzero(as_tuple=True)
            if not len(token):
                continue
            first = _product(x[token], gate_up[expert * 2 * inter:(expert + 1) * 2 * inter], fmt, math_name, tops[0])
            gate, up = first[:, :inter], first[:, inter:]
            middle = (gate / (1.0 + torch.exp(-gate)) * up).to(torch.bfloat16)
            last = _product(middle, down[expert * latent:(expert + 1) * latent], fmt, math_name, tops[1])
            out.index_add_(0, token, last * weights[token, slot].unsqueeze(1))
        outputs += [None, weights, entropy, confidence, out]
    return outputs

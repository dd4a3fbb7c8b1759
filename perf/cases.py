"""The work that a program using this library has it do, as measurable cases.

Sizes are those of the repository's own workloads (bench.py: the 4096-wide hybrid stack, the 2688-wide MoE layer
with 128 experts of 1856 and a 3712-wide shared expert) and generic ragged ones.  A serving program keeps, per
layer, its tiled weights, scales, workspace and output buffers, and calls the C ABI on them; decode cases walk
several layers of distinct weights, as a decode step does, so that no cache serves the weights of the next pass.
"""
import ctypes
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "nemotron-cutile-rs_amd"))

import nemotron_hip as NH  # noqa: E402

DT = {"f32": (torch.float32, NH.F32), "bf16": (torch.bfloat16, NH.BF16)}
_context = None


def context():
    """The program's one library context."""
    global _context
    if _context is None:
        _context = NH.Context(0)
    return _context


def listed():
    return [
        # the dequant GEMV of one f32 row: the smallest call, launch and latency bound
        {"name": "w8a32_m1", "op": "w8a32", "m": 1, "k": 4096, "n": 4096, "layers": 1},
        # single-stream decode: the SSM in_proj layers of a step, one token
        {"name": "linear_m1_in", "op": "linear", "m": 1, "k": 4096, "n": 16384, "layers": 6, "x": "bf16", "out": "bf16",
         "bias": False},
        # batch-8 decode: the out_proj layers of a step, with biases
        {"name": "linear_m8_out", "op": "linear", "m": 8, "k": 8192, "n": 4096, "layers": 10, "x": "bf16",
         "out": "bf16", "bias": True},
        # a serving batch of 77 sequences: the qkv projections of a step
        {"name": "linear_m77_qkv", "op": "linear", "m": 77, "k": 4096, "n": 6144, "layers": 12, "x": "bf16",
         "out": "bf16", "bias": False},
        # prefill of 2048 tokens: the widest projection
        {"name": "linear_m2048_up", "op": "linear", "m": 2048, "k": 4096, "n": 21504, "layers": 1, "x": "bf16",
         "out": "bf16", "bias": False},
        # a ragged f32 prompt through a layer of odd width, f32 out (the reference's own row type)
        {"name": "linear_m613_f32", "op": "linear", "m": 613, "k": 2688, "n": 4099, "layers": 1, "x": "f32",
         "out": "f32", "bias": True},
        # single-stream decode through MLP layers (up, ReLU^2, down)
        {"name": "mlp_m1", "op": "mlp", "m": 1, "hidden": 4096, "inter": 21504, "layers": 2, "x": "bf16",
         "out": "bf16", "bias": False},
        # a 500-token prompt through an MLP layer
        {"name": "mlp_m500", "op": "mlp", "m": 500, "hidden": 4096, "inter": 21504, "layers": 1, "x": "bf16",
         "out": "bf16", "bias": False},
        # batch-8 decode through the MoE layer from its input: router, 128 experts top-6, shared expert
        {"name": "moe_t8", "op": "moe", "tokens": 8, "hidden": 2688, "inter": 1856, "experts": 128, "top_k": 6,
         "shared": 3712, "x": "bf16", "out": "bf16"},
        # a 512-token prompt through the same layer
        {"name": "moe_t512", "op": "moe", "tokens": 512, "hidden": 2688, "inter": 1856, "experts": 128, "top_k": 6,
         "shared": 3712, "x": "bf16", "out": "bf16"},
        # INT4 weights: batch-4 decode
        {"name": "w4a8_m4", "op": "w4a8", "m": 4, "k": 4096, "n": 16384, "layers": 10, "x": "bf16", "out": "bf16",
         "bias": False},
        # INT4 weights: a 300-token prompt
        {"name": "w4a8_m300", "op": "w4a8", "m": 300, "k": 4096, "n": 16384, "layers": 1, "x": "bf16", "out": "bf16",
         "bias": False},
    ]


MAX_FLOPS = 3.6e11          # the listed prefill's
MAX_WEIGHTS = 384 << 20     # bytes of weights walked by a decode pass
MAX_MOE_WEIGHTS = 1.27e9


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A K width: whole 16s (the device envelope), half of them whole 512s."""
    v = _log(rng, lo, hi)
    return max(512, v // 512 * 512) if v >= 512 and rng.random() < 0.5 else max(16, v // 16 * 16)


def _layers(rng, m, weight_bytes):
    if m > 128 or rng.random() < 0.2:
        return 1
    return max(1, min(12, int(MAX_WEIGHTS // weight_bytes)))


def draw(rng):
    while True:
        op = rng.choices(["linear", "mlp", "moe", "w4a8", "w8a32"], [45, 15, 20, 12, 8])[0]
        x = "f32" if rng.random() < 0.25 else "bf16"
        out = "f32" if rng.random() < 0.3 else "bf16"
        bias = rng.random() < 0.4
        if op in ("linear", "w4a8"):
            m, k, n = _log(rng, 1, 2048), _width(rng, 256, 21504), _log(rng, 256, 21504)
            if rng.random() < 0.5:
                n = max(64, n // 64 * 64)
            wb = n * k if op == "linear" else n * k // 2
            case = {"op": op, "m": m, "k": k, "n": n, "layers": _layers(rng, m, wb), "x": x, "out": out, "bias": bias}
        elif op == "w8a32":
            m, k, n = _log(rng, 1, 16), _width(rng, 256, 8192), _log(rng, 256, 16384)
            case = {"op": op, "m": m, "k": k, "n": n, "layers": _layers(rng, m, n * k)}
        elif op == "mlp":
            m, hidden, inter = _log(rng, 1, 1024), _width(rng, 256, 4096), _width(rng, 512, 21504)
            case = {"op": op, "m": m, "hidden": hidden, "inter": inter, "layers": _layers(rng, m, 2 * hidden * inter),
                    "x": x, "out": out, "bias": bias}
        else:
            experts = rng.choice([8, 16, 60, 64, 128])
            case = {"op": op, "tokens": _log(rng, 1, 768), "hidden": _width(rng, 512, 4096),
                    "inter": _width(rng, 256, 1856), "experts": experts, "top_k": rng.randint(1, 8),
                    "shared": _width(rng, 512, 4096) if rng.random() < 0.6 else 0, "x": x, "out": out}
            if experts * case["hidden"] * case["inter"] * 2 > MAX_MOE_WEIGHTS:
                continue
        if work(case)["flops"] <= MAX_FLOPS:
            return case


# ---- inputs (torch alone) -------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _shapes(case):
    """[(n, k)] of each layer's weight matrices."""
    if case["op"] == "mlp":
        return [(case["inter"], case["hidden"]), (case["hidden"], case["inter"])]
    return [(case["n"], case["k"])]


def _normal(gen, shape, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(dtype)


def _rows(case, gen):
    return _normal(gen, (case.get("m") or case["tokens"], case.get("k") or case["hidden"]),
                   dtype=DT[case.get("x", "f32")][0])


def _dense_inputs(case, seed):
    """Per layer: the rows, the f32 weights (int4: the packed codes) and the biases."""
    gen = _generator(seed)
    for _ in range(case["layers"]):
        x = _rows(case, gen)
        if case["op"] == "w4a8":
            ws = [torch.randint(0, 256, ((case["k"] * case["n"] + 1) // 2,), generator=gen, device="cuda",
                                dtype=torch.uint8)]
        else:
            ws = [_normal(gen, s, 0.02) for s in _shapes(case)]
        bs = [_normal(gen, (s[0],), 0.1) if case.get("bias") else None for s in _shapes(case)]
        yield x, ws, bs


INT4_SCALE, INT4_ZERO = 0.0125, 8


class _MoeInputs:
    def __init__(self, case, seed):
        self.case, self.gen = case, _generator(seed)
        self.x = _rows(case, self.gen)
        self.router_w = _normal(self.gen, (case["hidden"], case["experts"]), 0.02)
        self.router_b = _normal(self.gen, (case["experts"],), 0.1)

    def experts(self):
        """The f32 up and down weights of each expert, then of the shared one."""
        h, i, s = (self.case[k] for k in ("hidden", "inter", "shared"))
        for _ in range(self.case["experts"]):
            yield _normal(self.gen, (i, h), 0.02), _normal(self.gen, (h, i), 0.02)
        if s:
            yield _normal(self.gen, (s, h), 0.02), _normal(self.gen, (h, s), 0.02)


# ---- what a program keeps -------------------------------------------------

class Bound:
    """Entry points with their arguments bound, as a serving loop keeps them."""

    def __init__(self):
        self.err = NH.NhError()
        self.calls, self.keep, self.outs = [], [], []

    def add(self, name, *args):
        fn = getattr(NH.lib(), name)
        simple = (ctypes.c_size_t, ctypes.c_int, ctypes.c_float, ctypes.c_uint32, ctypes.c_void_p)
        conv = [t(a) if t in simple and not isinstance(a, t) else a for t, a in zip(fn.argtypes, args)]
        self.calls.append((fn, (*conv, ctypes.byref(self.err))))

    def hold(self, t):
        self.keep.append(t)
        return None if t is None else t.data_ptr()


def _bytes(n):
    return torch.empty(max(int(n), 16), dtype=torch.uint8, device="cuda")


def _int8_weights(w):
    """f32 [n][k] -> (tiled int8 codes, f32 scales), through the library's offline path."""
    n, k = w.shape
    ctx = context().handle
    q, s = torch.empty((n, k), dtype=torch.int8, device="cuda"), torch.empty(n, device="cuda")
    t = _bytes(NH.lib().nh_tiled_weights_bytes(n, k))
    stream = torch.cuda.current_stream().cuda_stream
    NH.call("nh_quantize_rows_i8", ctx, w.data_ptr(), NH.F32, n, k, q.data_ptr(), s.data_ptr(), None, stream)
    NH.call("nh_tile_weights_i8", ctx, q.data_ptr(), n, k, t.data_ptr(), t.numel(), stream)
    return t, s


def _prepare_dense(case, seed):
    b, lib, ctx = Bound(), NH.lib(), context().handle
    stream = torch.cuda.current_stream().cuda_stream
    op, m = case["op"], case["m"]
    flag = b.hold(torch.zeros(1, dtype=torch.int64, device="cuda"))  # the non-finite word
    ws = None
    for x, weights, biases in _dense_inputs(case, seed):
        px, pb = b.hold(x), [b.hold(t) for t in biases]
        if op == "w4a8":
            n, k = case["n"], case["k"]
            w4 = _bytes(lib.nh_tiled_int4_weights_bytes(n, k))
            NH.call("nh_tile_weights_int4", ctx, weights[0].data_ptr(), weights[0].numel(), k, n, INT4_ZERO,
                    w4.data_ptr(), w4.numel(), stream)
            pw = [(b.hold(w4), None)]
        else:
            pw = [tuple(b.hold(t) for t in _int8_weights(w)) for w in weights]
        out = torch.empty((m, case.get("n") or case["hidden"]), dtype=DT[case.get("out", "f32")][0], device="cuda")
        b.outs.append(out)
        po, xd, od = out.data_ptr(), DT[case.get("x", "f32")][1], DT[case.get("out", "f32")][1]
        if ws is None:  # one workspace: the layers run one after another
            need = {"linear": lambda: lib.nh_linear_w8a8_workspace_size(m, case["k"]),
                    "mlp": lambda: lib.nh_mlp_w8a8_workspace_size(m, case["hidden"], case["inter"]),
                    "w4a8": lambda: lib.nh_linear_w4a8_workspace_size(m, case["n"], case["k"]),
                    "w8a32": lambda: 0}[op]()
            t = _bytes(need)
            b.hold(t)
            ws = (t.data_ptr(), t.numel())
        if op == "linear":
            b.add("nh_linear_w8a8", ctx, px, xd, *pw[0], pb[0], m, case["n"], case["k"], po, od, *ws, None, None, flag,
                  stream)
        elif op == "mlp":
            b.add("nh_mlp_w8a8", ctx, px, xd, *pw[0], pb[0], *pw[1], pb[1], m, case["hidden"], case["inter"], po, od,
                  *ws, flag, stream)
        elif op == "w4a8":
            b.add("nh_linear_w4a8", ctx, px, xd, pw[0][0], INT4_SCALE, INT4_ZERO, pb[0], m, case["n"], case["k"], po,
                  od, *ws, flag, stream)
        else:
            b.add("nh_gemv_w8a32", ctx, px, *pw[0], m, case["n"], case["k"], po, stream)
    return b


def _prepare_moe(case, seed):
    b, lib, ctx = Bound(), NH.lib(), context().handle
    stream = torch.cuda.current_stream().cuda_stream
    t, h, i, e, k, s = (case[v] for v in ("tokens", "hidden", "inter", "experts", "top_k", "shared"))
    inputs = _MoeInputs(case, seed)
    px, prw, prb = b.hold(inputs.x), b.hold(inputs.router_w), b.hold(inputs.router_b)
    ups, downs = [], []
    for up, down in inputs.experts():
        ups.append(_int8_weights(up))
        downs.append(_int8_weights(down))
    shared = [None] * 4
    if s:
        shared = [b.hold(v) for v in (*ups.pop(), *downs.pop())]
    pw = []
    for ws in (ups, downs):  # the experts back to back
        pw += [b.hold(torch.cat([w for w, _ in ws])), b.hold(torch.cat([v for _, v in ws]))]
    out = torch.empty((t, h), dtype=DT[case["out"]][0], device="cuda")
    b.outs.append(out)
    ws = _bytes(lib.nh_moe_layer_w8a8_workspace_size(t, h, i, e, k, s))
    flag = b.hold(torch.zeros(1, dtype=torch.int64, device="cuda"))
    b.add("nh_moe_layer_w8a8", ctx, px, DT[case["x"]][1], prw, prb, t, h, i, e, k, 1, 1.0, *pw, s, *shared, None,
          out.data_ptr(), DT[case["out"]][1], b.hold(ws), ws.numel(), flag, stream)
    return b


def prepare(case, seed):
    return _prepare_moe(case, seed) if case["op"] == "moe" else _prepare_dense(case, seed)


def run(state):
    for fn, args in state.calls:
        status = fn(*args)
        if status:
            NH.check(status, state.err)
    return state.outs


# ---- cost and expected values ---------------------------------------------

def work(case):
    """Weights, scales, rows and outputs once each; the multiply-adds of the products."""
    size = {"f32": 4, "bf16": 2}
    xs, os_ = size[case.get("x", "f32")], size[case.get("out", "f32")]
    if case["op"] == "moe":
        t, h, i, e, k, s = (case[v] for v in ("tokens", "hidden", "inter", "experts", "top_k", "shared"))
        touched = e * (1 - (1 - k / e) ** t)  # experts that receive a route
        weights = touched * (2 * h * i + 4 * (h + i)) + (2 * h * s + 4 * (h + s) if s else 0)
        return {"bytes": weights + 4 * h * e + 4 * e + t * h * (xs + os_),
                "flops": 2.0 * t * h * (2 * k * i + 2 * s + e)}
    m, w4 = case["m"], case["op"] == "w4a8"
    shapes = _shapes(case)
    bias = 4 if case.get("bias") else 0
    weights = sum((n * k // 2 if w4 else n * k + 4 * n) + bias * n for n, k in shapes)
    rows = m * (xs * shapes[0][1] + os_ * shapes[-1][0])
    return {"bytes": float(case["layers"] * (weights + rows)),
            "flops": 2.0 * case["layers"] * m * sum(n * k for n, k in shapes)}


def tolerance(case):
    # Codes and integer sums are exact, so what is left is the order of the scale products and sums in 32 bits, and
    # the rounding to the output type: errors against exact() measured 1.2e-7 in f32 and 1.7e-3 in bf16.  Layers
    # that quantize an intermediate can also see one of its codes fall to the other side of a tie: 2.2e-5 of the
    # whole at 300 tokens, so up to 4e-4 at one.
    if case.get("out") == "bf16":
        return {"rel": 7e-3, "max": 2e-2}
    return {"rel": 2e-3, "max": 2e-2} if case["op"] in ("mlp", "moe") else {"rel": 2e-6, "max": 1e-4}


def _quantize(x):
    """Symmetric int8 rows: (codes as f64, f32 scales as f64)."""
    x = x.to(torch.float32)
    s = (x.abs().amax(dim=1).double() / 127.0).to(torch.float32).double()
    v = (x.double() / s.clamp(min=1e-300)[:, None]).to(torch.float32).double()
    r = torch.trunc(v)
    r = (r + torch.where((v - r).abs() >= 0.5, torch.sign(v), torch.zeros_like(v))).clamp(-127, 127)
    return torch.where(s[:, None] > 0, r, torch.zeros_like(r)), s


def _linear(x, w):
    xq, sx = _quantize(x)
    wq, sw = w
    return (xq @ wq.T) * sx[:, None] * sw[None, :]


def _mlp(x, up, down, b_up=None, b_down=None):
    h = _linear(x, up)
    h = h if b_up is None else h + b_up.double()
    y = _linear(h.clamp(min=0).square(), down)
    return y if b_down is None else y + b_down.double()


def _exact_moe(case, seed):
    inputs = _MoeInputs(case, seed)
    x, e, k = inputs.x, case["experts"], case["top_k"]
    logits = (x.double() @ inputs.router_w.double() + inputs.router_b.double()).to(torch.float32).double()
    w, idx = torch.sigmoid(logits).topk(k, dim=1)
    w = w / w.sum(dim=1, keepdim=True)
    out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for n, (up, down) in enumerate(inputs.experts()):
        up, down = _quantize(up), _quantize(down)
        if n == e:  # the shared expert takes every row
            out += _mlp(x, up, down)
            continue
        t, j = (idx == n).nonzero(as_tuple=True)
        if t.numel():
            out[t] += w[t, j][:, None] * _mlp(x[t], up, down)
    return [out]


def exact(case, seed):
    if case["op"] == "moe":
        return _exact_moe(case, seed)
    outs = []
    for x, ws, bs in _dense_inputs(case, seed):
        if case["op"] == "mlp":
            outs.append(_mlp(x, _quantize(ws[0]), _quantize(ws[1]), *bs))
            continue
        n, k = case["n"], case["k"]
        if case["op"] == "w4a8":
            p = ws[0]
            codes = torch.stack([p & 15, p >> 4], dim=1).reshape(-1)[: k * n].reshape(k, n)
            scale = torch.full((n,), INT4_SCALE, dtype=torch.float32, device="cuda").double()
            y = _linear(x, ((codes.double() - INT4_ZERO).T, scale))
        elif case["op"] == "w8a32":
            wq, sw = _quantize(ws[0])
            y = (x.double() @ wq.T) * sw[None, :]
        else:
            y = _linear(x, _quantize(ws[0]))
        outs.append(y if bs[0] is None else y + bs[0].double())
    return outs

"""Performance cases of the fused KAN kernels on one MI355X.

Each case is one call (or one training step) that a program built on ``metal_kans`` makes again and
again, through the package's public entry points:

* ``layer``  -- inference of one layer on GPU tensors (``TorchMetalKANLinear`` under ``no_grad``):
                Chebyshev / RBF / B-spline, fp32 / fp16 / bf16;
* ``mlp``    -- inference of a small network (``TorchMetalKAN``), activations between layers in fp32;
* ``train``  -- one training step of a Chebyshev layer: forward, backward, in-place SGD update
                (so the next forward meets changed weights);
* ``gated``  -- the quantized GatedKAN block (``kans_gated_forward`` on device arrays): decode at up
                to 32 rows, prefill above, INT8 / INT4 / ternary weights;
* ``host``   -- the NumPy API (``ChebyKAN.__call__``): host array in, host array out.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what the
program holds before the call, ``run`` is the call, ``work`` its least traffic and arithmetic,
``tolerance`` what another correct implementation of the same precision may differ by and ``exact``
the same results in 64 bits.

GPU tensors live on a stream of their own (``torch.cuda.stream``), which the package launches on.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "metal-kans_amd"))

import metal_kans as mk  # noqa: E402

TORCH_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
LR = 1e-4

_LISTED = [
    # the smallest layer call: one hidden layer of a tabular network on one batch; launch latency counts
    {"name": "layer_cheby_f32_256x64x64", "kind": "layer", "basis": "cheby", "dtype": "f32", "B": 256, "d_in": 64,
     "d_out": 64, "degree": 9},
    # a wide RBF layer on normalised activations in half precision (an MLP replacement in a transformer)
    {"name": "layer_rbf_f16_16384x1024", "kind": "layer", "basis": "rbf", "dtype": "f16", "B": 16384, "d_in": 1024,
     "d_out": 1024, "degree": 8},
    # the classic KAN layer in full precision, expanding fourfold: the largest forward here
    {"name": "layer_bspline_f32_8192x1024x4096", "kind": "layer", "basis": "bspline", "dtype": "f32", "B": 8192,
     "d_in": 1024, "d_out": 4096, "degree": 5},
    # a ragged layer: no dimension a multiple of a tile
    {"name": "layer_cheby_bf16_3001x777x1300", "kind": "layer", "basis": "cheby", "dtype": "bf16", "B": 3001,
     "d_in": 777, "d_out": 1300, "degree": 5},
    # the digit classifier 784 -> 256 -> 256 -> 10 with half-precision weights, one evaluation batch
    {"name": "mlp_cheby_f16_4096x784", "kind": "mlp", "dtype": "f16", "B": 4096, "dims": "784,256,256,10",
     "degree": 9},
    # one training step of a small layer (function fitting, tabular data): latency counts
    {"name": "train_cheby_f32_256x64x64", "kind": "train", "dtype": "f32", "B": 256, "d_in": 64, "d_out": 64,
     "degree": 9},
    # one training step of a wide layer at the default degree
    {"name": "train_cheby_f32_8192x1024", "kind": "train", "dtype": "f32", "B": 8192, "d_in": 1024, "d_out": 1024,
     "degree": 4},
    # one training step with 16-bit parameters and ragged sizes
    {"name": "train_cheby_bf16_2000x300x500", "kind": "train", "dtype": "bf16", "B": 2000, "d_in": 300, "d_out": 500,
     "degree": 6},
    # one token through a quantized transformer-sized block
    {"name": "gated_int4_b1", "kind": "gated", "fmt": "int4", "B": 1, "d": 4096, "h": 11008},
    # a batch of decoding sequences through the same block in ternary weights
    {"name": "gated_ternary_b32", "kind": "gated", "fmt": "ternary", "B": 32, "d": 4096, "h": 11008},
    # a prompt of 512 tokens through the block
    {"name": "gated_int4_b512", "kind": "gated", "fmt": "int4", "B": 512, "d": 4096, "h": 11008},
    # the NumPy API at the size class the package is first met with
    {"name": "host_cheby_f32_4096x64x64", "kind": "host", "basis": "cheby", "dtype": "f32", "B": 4096, "d_in": 64,
     "d_out": 64, "degree": 4},
]

# no drawn case is larger than the largest listed one
_MOST_FLOPS = {"layer": 6e11, "train": 2.4e11, "gated": 6e11, "host": 5e9}


def listed():
    return [dict(c) for c in _LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size spread over the logarithm of the range: as it comes, or rounded to a multiple of 8 / 64."""
    v = _log_int(rng, lo, hi)
    m = rng.choice((1, 8, 64))
    return max(lo, min(hi, v // m * m))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "train", "train", "train", "gated", "gated", "gated", "mlp", "host"))
    while True:
        if kind == "layer":
            c = {"kind": kind, "basis": rng.choice(("cheby", "rbf", "bspline")),
                 "dtype": rng.choice(("f32", "f16", "bf16")), "B": _size(rng, 64, 16384),
                 "d_in": _size(rng, 16, 2048), "d_out": _size(rng, 16, 4096), "degree": rng.randint(3, 9)}
            if c["basis"] == "bspline":
                c["degree"] = rng.randint(2, 7)
        elif kind == "train":
            c = {"kind": kind, "dtype": rng.choice(("f32", "f32", "bf16", "f16")), "B": _size(rng, 64, 8192),
                 "d_in": _size(rng, 16, 2048), "d_out": _size(rng, 16, 2048), "degree": rng.randint(2, 10)}
        elif kind == "gated":
            decode = rng.random() < 0.5
            d = rng.choice((1024, 2048, 2560, 4096))
            c = {"kind": kind, "fmt": rng.choice(("int4", "int8", "ternary")),
                 "B": rng.randint(1, 32) if decode else _log_int(rng, 33, 1024), "d": d,
                 "h": rng.choice((d * 11 // 4, d * 43 // 16, d * 3 + 40))}
        elif kind == "mlp":
            dims = [_size(rng, 16, 784), _size(rng, 32, 512), _size(rng, 32, 512), rng.randint(2, 100)]
            c = {"kind": kind, "dtype": rng.choice(("f16", "f32")), "B": _size(rng, 64, 8192),
                 "dims": ",".join(map(str, dims)), "degree": rng.randint(4, 9)}
        else:
            c = {"kind": kind, "basis": rng.choice(("cheby", "rbf", "bspline")), "dtype": rng.choice(("f32", "f16")),
                 "B": _size(rng, 64, 8192), "d_in": _size(rng, 16, 256), "d_out": _size(rng, 16, 256),
                 "degree": rng.randint(4, 8)}
        if work(c)["flops"] <= _MOST_FLOPS.get(kind, 6e11):
            return c


# ---- sizes ---------------------------------------------------------------------------------------

def _slots(case):
    """Basis functions per feature and the base branch."""
    return case["degree"] + (3 if case.get("basis") == "bspline" else 0) + 1


def _esize(dt):
    return 4 if dt == "f32" else 2


def _gated_bytes(fmt, d_out, kd):
    if fmt == "ternary":
        return d_out * ((kd + 15) // 16 * 4 + (kd + 31) // 32 * 4)
    g = d_out * ((kd + 63) // 64)
    return g * ((32 if fmt == "int4" else 64) + 8)


def work(case):
    """Bytes: each input, weight and output once, in the element type the call hands over; flops: the
    dense contraction over features and basis functions (the basis values themselves left out)."""
    B, kind = case["B"], case["kind"]
    if kind in ("layer", "host"):
        e = _esize(case["dtype"])
        n = case["d_in"] * case["d_out"] * _slots(case)
        return {"bytes": e * (B * (case["d_in"] + case["d_out"]) + n + case["d_out"]), "flops": 2 * B * n}
    if kind == "mlp":
        dims, e = [int(v) for v in case["dims"].split(",")], _esize(case["dtype"])
        n = sum(a * b for a, b in zip(dims, dims[1:])) * _slots(case)
        return {"bytes": 4 * B * (dims[0] + dims[-1]) + e * (n + sum(dims[1:])), "flops": 2 * B * n}
    if kind == "train":
        e = _esize(case["dtype"])
        n = case["d_in"] * case["d_out"] * _slots(case)
        # x, dy read, y, dx written; weights read and updated, their gradients written
        return {"bytes": e * (2 * B * (case["d_in"] + case["d_out"]) + 3 * (n + case["d_out"])), "flops": 6 * B * n}
    d, h = case["d"], case["h"]
    b = sum(_gated_bytes(case["fmt"], o, kd) for o, i in ((h, d), (h, d), (d, h)) for kd in (4 * i, i))
    return {"bytes": b + 4 * B * d, "flops": 2 * B * 3 * d * h * 5}


def tolerance(case):
    """fp32: sums in another order; fp16 / bf16: operands and results rounded to 16 bits.  About four times
    the error measured against 64 bits: fp32 1.7e-6, fp16 3e-4, bf16 2e-3 to 2.4e-3, quantized blocks 8e-4,
    the fp16 network 3.7e-3."""
    kind = case["kind"]
    if kind == "gated":
        return {"rel": 4e-3, "max": 0.1}
    if kind == "mlp":
        # three layers of nine coefficients amplify the rounding of 16-bit operands (T_k'(1) = k^2)
        return {"rel": 1.5e-2, "max": 0.5} if case["dtype"] == "f16" else {"rel": 1e-5, "max": 4e-4}
    return {"f32": {"rel": 6e-6, "max": 2e-4}, "f16": {"rel": 2e-3, "max": 0.08},
            "bf16": {"rel": 1e-2, "max": 0.4}}[case["dtype"]]


# ---- inputs --------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _layer_weights(g, d_in, d_out, K, dt):
    """Weights as a layer starts training: uniform in +-1/sqrt(d_in); a bias that training has moved."""
    b = 1.0 / math.sqrt(d_in)

    def u(*shape):
        return ((torch.rand(*shape, generator=g, device="cuda") * 2 - 1) * b).to(TORCH_DT[dt])
    return u(d_out, d_in * K), u(d_out, d_in), u(d_out)


def _layer_input(g, basis, B, d_in, dt):
    """Chebyshev layers meet activations that mostly lie in [-1, 1], B-splines some outside their grid,
    RBF layers normalised ones."""
    if basis == "cheby":
        x = torch.tanh(torch.randn(B, d_in, generator=g, device="cuda"))
        x *= 1.05
    elif basis == "bspline":
        x = torch.rand(B, d_in, generator=g, device="cuda") * 2.4 - 1.2
    else:
        x = torch.randn(B, d_in, generator=g, device="cuda")
        x = (x - x.mean(1, keepdim=True)) / x.std(1, keepdim=True)
    return x.to(TORCH_DT[dt])


def _layer_inputs(case, seed):
    g = _gen(seed)
    K = _slots(case) - 1
    basis = case.get("basis", "cheby")
    ws = _layer_weights(g, case["d_in"], case["d_out"], K, case["dtype"])
    x = _layer_input(g, basis, case["B"], case["d_in"], case["dtype"])
    dy = (torch.randn(case["B"], case["d_out"], generator=g, device="cuda") / case["B"]).to(x.dtype)
    return x, ws, dy


def _fill(module, ws):
    with torch.no_grad():
        for p, w in zip((module.weight, module.base_weight, module.bias_param), ws):
            p.copy_(w)


def _mlp_inputs(case, seed):
    g = _gen(seed)
    dims = [int(v) for v in case["dims"].split(",")]
    # weights ~ N(0, 1 / (d_in K)), which keeps the activations near the domain
    ws = []
    for a, b in zip(dims, dims[1:]):
        w = torch.randn(b, a * case["degree"], generator=g, device="cuda") / math.sqrt(a * case["degree"])
        wb = torch.randn(b, a, generator=g, device="cuda") / math.sqrt(a)
        ws.append([t.to(TORCH_DT[case["dtype"]]) for t in (w, 0.5 * wb, 0.1 * wb[:, 0].contiguous())])
    return torch.rand(case["B"], dims[0], generator=g, device="cuda"), ws


def _gated_codes(g, fmt, d_out, kd):
    """Codes and group parameters of weights ~ N(0, 0.02): (codes [d_out][padded], per-group scale, bias)."""
    grp = 32 if fmt == "ternary" else 64
    pad = (kd + grp - 1) // grp * grp
    z = torch.randn(d_out, pad, generator=g, device="cuda")
    var = 1.0 + 0.1 * torch.randn(d_out * (pad // grp), generator=g, device="cuda").clamp_(-3, 3)
    if fmt == "ternary":
        q = (z * 1.25).round_().clamp_(-1, 1).add_(1).to(torch.uint8)
        q[:, kd:] = 0
        return q, 0.016 * var, None
    top = 15 if fmt == "int4" else 255
    q = ((z / 4.8 + 0.5) * top).round_().clamp_(0, top).to(torch.uint8)
    scale = 0.02 * 4.8 / top * var
    return q, scale, -0.5 * top * scale


def _gated_packed(fmt, q, kd):
    """Codes in the packed layout of the quantized weight formats."""
    if fmt == "int8":
        return q
    if fmt == "int4":
        p = q.view(q.shape[0], -1, 2)
        return p[:, :, 0] | (p[:, :, 1] << 4)
    w = (kd + 15) // 16
    p = q[:, : w * 16].reshape(q.shape[0], w * 4, 4)
    return p[:, :, 0] | (p[:, :, 1] << 2) | (p[:, :, 2] << 4) | (p[:, :, 3] << 6)


def _gated_x(case, seed):
    x = torch.randn(case["B"], case["d"], generator=_gen(seed), device="cuda")
    return (0.4 * x).to(torch.float16)


def _gated_matrices(case, seed):
    """(d_out, kd) of the six matrices (gate, up, down; basis and base weights) and their generators."""
    d, h = case["d"], case["h"]
    for j, (o, i) in enumerate(((h, d), (h, d), (d, h))):
        for m, kd in enumerate((4 * i, i)):
            yield j, m, o, kd, _gen(seed * 64 + 2 * j + m + 1)


# ---- prepare / run -------------------------------------------------------------------------------

class _Block:
    """A quantized GatedKAN block on the device (handles freed with the state)."""

    def __init__(self, case, seed):
        self.lib = mk.get_metal_bridge()
        fmt, K = case["fmt"], 4
        arrs = [[], [], []]
        for j, m, o, kd, g in _gated_matrices(case, seed):
            q, s, b = _gated_codes(g, fmt, o, kd)
            arrs[j].append(_gated_packed(fmt, q, kd).contiguous().cpu().numpy())
            arrs[j].append(s.cpu().numpy())
            if b is not None:
                arrs[j].append(b.cpu().numpy())
        d, h = case["d"], case["h"]
        create = {"int4": self.lib.kans_qlayer_create_int4, "int8": self.lib.kans_qlayer_create_int8,
                  "ternary": self.lib.kans_qlayer_create_ternary}[fmt]
        self.layers = []
        for (o, i), a in zip(((h, d), (h, d), (d, h)), arrs):
            p = ctypes.c_void_p()
            mk.device.check(create(i, o, K, 1, 0, 32 if fmt == "ternary" else 64, *[v.ctypes.data for v in a], None, 0,
                                   ctypes.byref(p)), "kans_qlayer_create")
            self.layers.append(p)
        self.handle = ctypes.c_void_p()
        mk.device.check(self.lib.kans_gated_create(*self.layers, ctypes.byref(self.handle)), "kans_gated_create")

    def __del__(self):
        self.lib.kans_gated_destroy(self.handle)
        for p in self.layers:
            self.lib.kans_qlayer_destroy(p)


_STREAM = None


def _stream():
    """The program's stream."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "stream": _stream()}
    with torch.cuda.stream(s["stream"]):
        if kind in ("layer", "train"):
            x, ws, dy = _layer_inputs(case, seed)
            m = mk.TorchMetalKANLinear(case["d_in"], case["d_out"], basis=case.get("basis", "cheby"),
                                       degree=case["degree"]).to("cuda").to(x.dtype)
            _fill(m, ws)
            s["module"], s["x"] = m, x
            if kind == "train":
                x.requires_grad_(True)
                s["dy"], s["params"] = dy, list(m.parameters())
        elif kind == "mlp":
            x, ws = _mlp_inputs(case, seed)
            dims = [int(v) for v in case["dims"].split(",")]
            net = mk.TorchMetalKAN(dims, degree=case["degree"]).to("cuda").to(TORCH_DT[case["dtype"]])
            for layer, w in zip(net.layers, ws):
                _fill(layer, w)
            s["module"], s["x"] = net, x
        elif kind == "gated":
            s["block"] = _Block(case, seed)
            s["x"] = _gated_x(case, seed)
            s["y"] = torch.empty_like(s["x"])
        else:
            x, ws, _ = _layer_inputs(case, seed)
            K = _slots(case) - 1
            cls = {"cheby": mk.ChebyKAN, "rbf": mk.FastKAN, "bspline": mk.BSplineKAN}[case["basis"]]
            layer = cls(case["d_in"], case["d_out"], case["degree"])
            attr = {"cheby": "w_cheby", "rbf": "w_rbf", "bspline": "w_spline"}[case["basis"]]
            for name, w in zip((attr, "w_base", "bias"), ws):
                setattr(layer, name, w.float().cpu().numpy())
            assert getattr(layer, attr).shape == (case["d_out"], case["d_in"] * K)
            if case["dtype"] == "f16":
                layer.half()
            s["layer"], s["x"] = layer, x.cpu().numpy()
    s["stream"].synchronize()
    return s


def run(state):
    kind = state["kind"]
    if kind == "host":
        return state["layer"](state["x"])
    with torch.cuda.stream(state["stream"]):
        if kind in ("layer", "mlp"):
            with torch.no_grad():
                return state["module"](state["x"])
        if kind == "train":
            x, params = state["x"], state["params"]
            x.grad = None
            for p in params:
                p.grad = None
            y = state["module"](x)
            y.backward(state["dy"])
            with torch.no_grad():
                for p in params:
                    p.add_(p.grad, alpha=-LR)
            return {"y": y.detach(), "dx": x.grad, "grads": [p.grad for p in params],
                    "params": [p.detach() for p in params]}
        x, y = state["x"], state["y"]
        d = x.shape[1]
        block = state["block"]
        f16 = 1
        mk.device.check(block.lib.kans_gated_forward(block.handle, x.data_ptr(), f16, d, y.data_ptr(), f16, d,
                                                     x.shape[0], 1, state["stream"].cuda_stream),
                        "kans_gated_forward")
        return y


# ---- the same in 64 bits -------------------------------------------------------------------------

def _basis(case, x, K):
    """phi_k(x) [B, d, K] in 64 bits."""
    basis = case.get("basis", "cheby")
    if basis == "cheby":
        t = x.clamp(-1, 1)
        out = [torch.ones_like(t), t]
        for _ in range(2, K):
            out.append(2 * t * out[-1] - out[-2])
        return torch.stack(out[:K], -1)
    if basis == "rbf":
        c = torch.from_numpy(np.linspace(-1.0, 1.0, K, dtype=np.float32)).double().to(x.device)
        if case["kind"] == "host" and case["dtype"] == "f16":
            c = c.half().double()     # a half-precision layer holds its centres in half precision
        h = 2.0 / (K - 1)
        return torch.exp(-(x[..., None] - c) ** 2 / (2 * h * h))
    G = K - 3
    pos = (x + 1.0) * (G / 2.0)
    span = pos.floor().clamp(0, G - 1)
    u = (pos - span).clamp(0, 1)
    w = ((1 - u) ** 3 / 6, (3 * u ** 3 - 6 * u ** 2 + 4) / 6, (-3 * u ** 3 + 3 * u ** 2 + 3 * u + 1) / 6, u ** 3 / 6)
    out = torch.zeros(*x.shape, K, dtype=x.dtype, device=x.device)
    for j in range(4):
        out.scatter_(-1, (span.long() + j)[..., None], w[j][..., None])
    return out


def _forward(case, x, W, Wb, b, K, rows=2048):
    """y in 64 bits, in blocks of rows (the expanded basis of a large batch does not fit otherwise)."""
    W, Wb = W.double(), Wb.double()
    out = []
    for xs in x.split(rows):
        xs = xs.double()
        y = _basis(case, xs, K).reshape(xs.shape[0], -1) @ W.T + (xs * torch.sigmoid(xs)) @ Wb.T
        out.append(y if b is None else y + b.double())
    return torch.cat(out)


def _exact_train(case, x, ws, dy, rows=2048):
    W, Wb, b = (w.double() for w in ws)
    K, d_in = case["degree"], case["d_in"]
    y = _forward(case, x, W, Wb, b, K)
    gW, gWb, dx = torch.zeros_like(W), torch.zeros_like(Wb), []
    for xs, g in zip(x.split(rows), dy.split(rows)):
        xs, g = xs.double(), g.double()
        sg = torch.sigmoid(xs)
        gW += g.T @ _basis(case, xs, K).reshape(xs.shape[0], -1)
        gWb += g.T @ (xs * sg)
        # T'_k by its own recurrence; zero where the input is clamped
        T, D = [torch.ones_like(xs), xs], [torch.zeros_like(xs), torch.ones_like(xs)]
        for _ in range(2, K):
            D.append(2 * T[-1] + 2 * xs * D[-1] - D[-2])
            T.append(2 * xs * T[-1] - T[-2])
        dphi = torch.stack(D[:K], -1) * ((xs >= -1) & (xs <= 1))[..., None]
        dx.append(((g @ W).reshape(xs.shape[0], d_in, K) * dphi).sum(-1) + (g @ Wb) * sg * (1 + xs * (1 - sg)))
    grads = [gW, gWb, dy.double().sum(0)]
    return {"y": y, "dx": torch.cat(dx), "grads": grads, "params": [w - LR * g for w, g in zip((W, Wb, b), grads)]}


def _exact_gated(case, seed):
    fmt = case["fmt"]
    x = _gated_x(case, seed)
    mats = [[None, None], [None, None], [None, None]]
    for j, m, o, kd, g in _gated_matrices(case, seed):
        q, s, b = _gated_codes(g, fmt, o, kd)
        grp = 32 if fmt == "ternary" else 64
        w = q.double().view(o, -1, grp)
        s = s.double().view(o, -1, 1)
        w = (w - 1) * s if b is None else w * s + b.double().view(o, -1, 1)
        mats[j][m] = w.view(o, -1)[:, :kd]
    act = {"basis": "cheby", "kind": "gated"}
    gate, up = (_forward(act, x, mats[j][0], mats[j][1], None, 4, rows=512) for j in (0, 1))
    hidden = gate * torch.sigmoid(gate) * up
    return _forward(act, hidden, mats[2][0], mats[2][1], None, 4, rows=512)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gated":
        return _exact_gated(case, seed)
    if kind == "mlp":
        x, ws = _mlp_inputs(case, seed)
        for W, Wb, b in ws:
            x = _forward(case, x, W, Wb, b, case["degree"])
        return x
    x, ws, dy = _layer_inputs(case, seed)
    if kind == "train":
        return _exact_train(case, x, ws, dy)
    y = _forward(case, x, *ws, _slots(case) - 1)
    return y.cpu().numpy() if kind == "host" else y

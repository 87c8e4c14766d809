"""The work that programs have these kernels do, as cases that can be timed and compared.

Every case goes through the public entry points: the four kernels of
cormorant_amd.kernels on device tensors, or an InferenceSession on an ONNX graph.
The sizes are those of the repository's graphs, benchmark and reference cases, or of
ordinary convolutional networks and matrix products; `draw` spreads over the ranges
between them, odd sizes among them.  Results are whole numbers (raw Q8.8) and have to
be the same bit for bit.

Activations are uniform or half-normal around one, weights normal with the variance
2 / fan-in that keeps a layer's output at its input's scale.  So some layers' weights
fit 8 bits and others' do not, as in trained networks.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cormorant_amd import kernels as K
from cormorant_amd import workloads as wl
from cormorant_amd.scheduler import InferenceSession, OnnxGraph, onnx_io

DEV = "cuda"
OPS = {"add": 0, "sub": 1, "mul": 2, "div": 3, "relu": 4, "relu6": 5}
POOLS = {"max": 0, "avg": 1, "lp": 2}
ACTS = {"none": 0, "relu": 1, "relu6": 2}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a classifier's single request: host arrays in, host arrays out, two small
        # products; launches, copies and waits are all there is
        {"name": "mlp_b64", "kind": "mlp", "batch": 64},
        # a whole image network at its serving batch, inputs already uploaded, logits
        # read back: 38 layers from 112x112 down to 7x7 planes
        {"name": "mobilenet_like_b16", "kind": "mobilenet", "batch": 16, "hw": 224},
        # a large dense layer: the largest product
        _matmul("matmul_4096", 1, 4096, 4096, 4096),
        # a dense layer whose sizes are multiples of nothing (vocabulary or class
        # counts are what they are), with a bias row and Relu
        _matmul("matmul_odd_2000x1283x1001", 1, 2000, 1283, 1001, add="column", act="relu"),
        # many small products in one call: a ragged token count per head
        _matmul("matmul_b96_196x64x196", 96, 196, 64, 196),
        # an early 3x3 layer of an image network, weights packed when the model is loaded
        _conv("conv_3x3_64to128_56", 32, 64, 56, 56, 128, 3, 1, 1, act="relu", packed=1),
        # a deep 3x3 layer: many channels, small planes, weights passed with each call
        _conv("conv_3x3_256_14", 32, 256, 14, 14, 256, 3, 1, 1, act="relu"),
        # the first layer of an image network: few channels, large window and planes
        _conv("conv_stem_7x7_s2", 16, 3, 224, 224, 64, 7, 2, 3, act="relu", packed=1),
        # a bottleneck's expansion: 1x1, with its residual Add and Relu
        _conv("conv_1x1_64to256_56", 32, 64, 56, 56, 256, 1, 1, 0, act="relu", add=1),
        # a depthwise layer of a mobile network on its large planes
        _conv("conv_dw_3x3_96_112", 32, 96, 112, 112, 96, 3, 1, 1, act="relu6", dw=1),
        # the pool behind an image network's first layer
        {"name": "pool_max_3x3_s2_112", "kind": "pool", "type": "max", "batch": 32, "ch": 64,
         "h": 112, "w": 112, "k": 3, "stride": 2, "pad": 1, "cip": 0},
        # one tensor against every image of a batch: subtracting the mean image
        {"name": "vectorop_sub_mean_256", "kind": "vectorop", "op": "sub", "size": 3 * 224 * 224,
         "outer": 256, "bcast": 1},
    ]


def _matmul(name, batch, n, k, m, add="none", act="none"):
    c = {"kind": "matmul", "batch": batch, "n": n, "k": k, "m": m, "add": add, "act": act}
    return dict(c, name=name) if name else c


def _conv(name, batch, ic, h, w, oc, k, stride, pad, dil=1, act="none", add=0, packed=0, dw=0):
    c = {"kind": "conv", "batch": batch, "ic": ic, "h": h, "w": w, "oc": oc, "k": k,
         "stride": stride, "pad": pad, "dil": dil, "act": act, "add": add, "packed": packed,
         "dw": dw}
    return dict(c, name=name) if name else c


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges:
    vectorop: every operation, 16 Ki to 48 Mi elements, flat or one operand repeated;
    matmul: batches of 1 to 128, n / k / m of 1 to 4096, 1 M to 30 G multiply-adds;
    conv: batches of 1 to 32, 3 to 512 channels, planes of 7 to 224, windows of 1, 3, 5
    and 7, strides 1 and 2, dilations 1 and 2, raw or packed weights, depthwise or not,
    1 M (depthwise) or 8 M to 4 G multiply-adds;
    pool: windows of 2, 3 or the whole plane, every kind, 256 Ki to 64 M elements;
    graphs: MLP batches of 1 to 256, the image network at 64 to 224 pixels, 1 to 16 images."""
    kind = rng.choice(["vectorop", "matmul", "matmul", "conv", "conv", "conv", "dw", "pool",
                       "pool", "mlp", "mobilenet"])
    if kind == "mlp":
        return {"kind": "mlp", "batch": _log(rng, 1, 256)}
    if kind == "mobilenet":
        return {"kind": "mobilenet", "batch": _log(rng, 1, 16), "hw": rng.choice([64, 96, 128, 160, 192, 224])}
    if kind == "vectorop":
        total = _log(rng, 1 << 14, 48 << 20)
        if rng.random() < 0.5:
            return {"kind": "vectorop", "op": rng.choice(sorted(OPS)), "size": total, "outer": 1, "bcast": 0}
        outer = min(_log(rng, 2, 256), max(2, total // 16))
        size = -(-total // outer)
        if rng.random() < 0.7:      # the scheduler rounds chunk strides up to 8 elements
            size = -(-size // 8) * 8
        return {"kind": "vectorop", "op": rng.choice(["add", "sub", "mul", "div"]), "size": size,
                "outer": outer, "bcast": 1}
    if kind == "matmul":
        while True:
            batch = 1 if rng.random() < 0.5 else _log(rng, 2, 128)
            n, k, m = (_log(rng, 1, 4096) for _ in range(3))
            if rng.random() < 0.5:
                n, k, m = (v if v < 16 else -(-v // 8) * 8 for v in (n, k, m))
            if 1 << 20 <= batch * n * k * m <= 30e9 and batch * (n * k + k * m + n * m) <= 100e6:
                return _matmul("", batch, n, k, m, add=rng.choice(["none", "none", "same", "column"]),
                               act=rng.choice(sorted(ACTS)))
    if kind == "pool":
        while True:
            h = _log(rng, 7, 224)
            w = h if rng.random() < 0.7 else _log(rng, 7, 224)
            k = rng.choice([2, 2, 3, 3, 3, 0])
            c = {"kind": "pool", "type": rng.choice(sorted(POOLS)), "batch": _log(rng, 1, 32),
                 "ch": _log(rng, 1, 1024), "h": h, "w": w, "k": k,
                 "stride": 1 if k == 0 else rng.choice([1, 2, 2]),
                 "pad": 0 if k < 3 else rng.choice([0, 1]), "cip": rng.choice([0, 1])}
            if 1 << 18 <= c["batch"] * c["ch"] * h * w <= 64e6:
                return c
    while True:
        h = _log(rng, 7, 224)
        w = h if rng.random() < 0.7 else _log(rng, 7, 224)
        k = rng.choice([3, 3, 5]) if kind == "dw" else rng.choice([1, 1, 3, 3, 3, 5, 7])
        dil = 2 if k == 3 and rng.random() < 0.2 else 1
        ic = _log(rng, 8 if kind == "dw" else 3, 512)
        oc = ic if kind == "dw" else _log(rng, 3, 512)
        if rng.random() < 0.6:
            ic, oc = (v if v < 8 else -(-v // 8) * 8 for v in (ic, oc))
        if kind == "dw":
            oc = ic
        c = _conv("", _log(rng, 1, 32), ic, h, w, oc, k, rng.choice([1, 1, 2]), dil * (k // 2), dil=dil,
                  act=rng.choice(sorted(ACTS)), add=rng.choice([0, 0, 1]), packed=rng.choice([0, 1]),
                  dw=int(kind == "dw"))
        oh, ow = _conv_out(c)
        macs = c["batch"] * oc * oh * ow * (1 if c["dw"] else ic) * k * k
        size = c["batch"] * (ic * h * w + oc * oh * ow)
        if 1 << (20 if c["dw"] else 23) <= macs <= 4e9 and size <= 64e6:
            return c


# ---------------------------------------------------------------- the inputs
def _gen(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _q88(x):
    """Real values to raw Q8.8: floor(256 x), saturated."""
    return torch.floor(x * 256.0).clamp_(-32768, 32767).to(torch.int16)


def _uniform(g, n, lo, hi):
    return _q88(torch.rand(n, generator=g, device=DEV) * (hi - lo) + lo)


def _normal(g, n, sigma):
    return _q88(torch.randn(n, generator=g, device=DEV) * sigma)


def _activations(g, n):
    """What a Relu leaves of a normal variable."""
    return _q88(torch.randn(n, generator=g, device=DEV).clamp_(min=0.0))


def _conv_out(c):
    return tuple((v + 2 * c["pad"] - c["dil"] * (c["k"] - 1) - 1) // c["stride"] + 1 for v in (c["h"], c["w"]))


def _pool_shape(c):
    """(kernel h, w, stride, pad, out h, out w); a window of 0 is the whole plane."""
    if c["k"] == 0:
        return c["h"], c["w"], 1, 0, 1, 1
    return (c["k"], c["k"], c["stride"], c["pad"],
            *((v + 2 * c["pad"] - c["k"]) // c["stride"] + 1 for v in (c["h"], c["w"])))


_models = {}   # graphs by their sizes: a program loads its model once


def _session(key, build):
    if key not in _models:
        _models[key] = onnx_io.encode_model(build())
    return InferenceSession(OnnxGraph(_models[key]))


def prepare(case, seed):
    g = _gen(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        s = _session(("mlp", case["batch"]), lambda: wl.mlp_model(case["batch"]))
        x = _uniform(g, case["batch"] * wl.MLP_IN, -1.0, 1.0).cpu().numpy().reshape(case["batch"], wl.MLP_IN)
        return {"case": case, "session": s, "x": x}
    if kind == "mobilenet":
        b, hw = case["batch"], case["hw"]
        s = _session(("mobilenet", b, hw), lambda: wl.mobilenet_model(b, hw))
        s.write_input("X", _uniform(g, b * 3 * hw * hw, -1.0, 1.0).cpu().numpy().reshape(b, 3, hw, hw))
        return {"case": case, "session": s}
    if kind == "vectorop":
        size, outer = case["size"], case["outer"]
        a = _uniform(g, size * outer, -8.0, 8.0)
        b = _uniform(g, size, -8.0, 8.0)
        if case["op"] == "div":
            b[b == 0] = 1
        return {"case": case, "a": a, "b": b, "c": torch.empty(size * outer, dtype=torch.int16, device=DEV)}
    if kind == "matmul":
        b, n, k, m = case["batch"], case["n"], case["k"], case["m"]
        st = {"case": case, "a": _normal(g, b * n * k, 1.0), "b": _normal(g, b * k * m, math.sqrt(2.0 / k)),
              "c": torch.empty(b * n * m, dtype=torch.int16, device=DEV), "add": None, "ws": None}
        if case["add"] != "none":
            st["add"] = _normal(g, m if case["add"] == "column" else b * n * m, 0.5)
        ws = K.matmul_workspace_size(n, k, m, *_matmul_strides(case))
        if ws:
            st["ws"] = torch.empty(ws, dtype=torch.uint8, device=DEV)
        return st
    if kind == "pool":
        _, _, _, _, oh, ow = _pool_shape(case)
        return {"case": case, "x": _uniform(g, case["batch"] * case["ch"] * case["h"] * case["w"], -4.0, 4.0),
                "y": torch.empty(case["batch"] * case["ch"] * oh * ow, dtype=torch.int16, device=DEV)}
    fan = (1 if case["dw"] else case["ic"]) * case["k"] ** 2
    oh, ow = _conv_out(case)
    out = case["batch"] * case["oc"] * oh * ow
    st = {"case": case, "x": _activations(g, case["batch"] * case["ic"] * case["h"] * case["w"]),
          "w": _normal(g, case["oc"] * fan, math.sqrt(2.0 / fan)), "b": _normal(g, case["oc"], 0.1),
          "y": torch.empty(out, dtype=torch.int16, device=DEV), "add": None, "ws": None, "packed": None}
    if case["add"]:
        st["add"] = _normal(g, out, 1.0)
    args = _conv_args(case)
    packed = K.conv_packed_size(*args) if case["packed"] else 0
    if packed:
        st["packed"] = torch.empty(packed, dtype=torch.uint8, device=DEV)
        K.conv_pack(st["w"], st["packed"], *args)
    else:
        ws = K.conv_workspace_size(*args)
        if ws:
            st["ws"] = torch.empty(ws, dtype=torch.uint8, device=DEV)
    return st


def _matmul_strides(c):
    return c["batch"], c["n"] * c["k"], c["k"] * c["m"], c["n"] * c["m"]


def _conv_args(c):
    oh, ow = _conv_out(c)
    return (c["batch"], c["ic"], c["h"], c["w"], c["oc"], oh, ow, c["k"], c["k"], c["stride"], c["stride"],
            c["dil"], c["dil"], c["pad"], c["pad"], 1, c["dw"])


# ------------------------------------------------------------------- one pass
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "mlp":
        return state["session"].run({"X": state["x"]})["Y"]
    if kind == "mobilenet":
        state["session"].launch()
        return state["session"].read_output("Y")
    if kind == "vectorop":
        bcast = c["bcast"]
        K.VectorOPKernel(state["a"], state["b"] if bcast or OPS[c["op"]] < 4 else None, state["c"], c["size"],
                         OPS[c["op"]], c["outer"], c["size"] if bcast else 0, 0)
        return state["c"]
    if kind == "matmul":
        K.MatmulKernel(state["a"], state["b"], state["c"], c["n"], c["k"], c["m"], *_matmul_strides(c),
                       add=state["add"], add_column=c["add"] == "column", act=ACTS[c["act"]],
                       workspace=state["ws"])
        return state["c"]
    if kind == "pool":
        kh, kw, s, p, oh, ow = _pool_shape(c)
        K.PoolingKernel(state["x"], state["y"], c["batch"], c["ch"], c["h"], c["w"], oh, ow, kh, kw, s, s, p, p,
                        1, 1, POOLS[c["type"]], 2, c["cip"])
        return state["y"]
    if state["packed"] is not None:
        K.ConvPackedKernel(state["x"], state["packed"], state["b"], state["y"], *_conv_args(c), add=state["add"],
                           act=ACTS[c["act"]])
    else:
        K.ConvKernel(state["x"], state["w"], state["b"], state["y"], *_conv_args(c), add=state["add"],
                     act=ACTS[c["act"]], workspace=state["ws"])
    return state["y"]


# ------------------------------------------------------- what a pass must do
def _mobilenet_layers(hw):
    """(in channels, out channels, window, out size) of every convolution."""
    s = wl.conv_out(hw, 3, 2, 1, 1)
    got, cin = [(3, 32, 3, s)], 32
    for cout, reps, stride in wl.MOBILENET_STAGES:
        for r in range(reps):
            s = wl.conv_out(s, 3, stride if r == 0 else 1, 1, 1)
            got += [(cin, cin, 3, s), (cin, cout, 1, s)]
            cin = cout
    return got + [(cin, wl.MOBILENET_HEAD, 1, s)]


def work(case):
    """Bytes: each input read once, each output written once.  Flops: two for each
    Q8.8 multiply-add (four 8-bit products of two 16-bit values, whatever the kernel
    issues), one for each element of the others."""
    kind = case["kind"]
    if kind == "mlp":
        w = wl.MLP_IN * wl.MLP_HIDDEN + wl.MLP_HIDDEN * wl.MLP_OUT
        return {"bytes": 2 * (w + case["batch"] * (wl.MLP_IN + wl.MLP_OUT)), "flops": 2 * case["batch"] * w}
    if kind == "mobilenet":
        layers = _mobilenet_layers(case["hw"])
        b, fc = case["batch"], wl.MOBILENET_HEAD * wl.MOBILENET_CLASSES
        weights = sum(i * o * k * k for i, o, k, _ in layers) + fc
        macs = b * (sum(i * o * k * k * s * s for i, o, k, s in layers) + fc)
        return {"bytes": 2 * (weights + b * (3 * case["hw"] ** 2 + wl.MOBILENET_CLASSES)), "flops": 2 * macs}
    if kind == "vectorop":
        n = case["size"] * case["outer"]
        return {"bytes": 2 * (2 * n + (case["size"] if OPS[case["op"]] < 4 else 0)), "flops": n}
    if kind == "matmul":
        b, n, k, m = case["batch"], case["n"], case["k"], case["m"]
        add = {"none": 0, "same": b * n * m, "column": m}[case["add"]]
        return {"bytes": 2 * (b * (n * k + k * m + n * m) + add), "flops": 2 * b * n * k * m}
    if kind == "pool":
        kh, kw, _, _, oh, ow = _pool_shape(case)
        planes = case["batch"] * case["ch"]
        return {"bytes": 2 * planes * (case["h"] * case["w"] + oh * ow), "flops": planes * oh * ow * kh * kw}
    oh, ow = _conv_out(case)
    fan = (1 if case["dw"] else case["ic"]) * case["k"] ** 2
    x, y = case["batch"] * case["ic"] * case["h"] * case["w"], case["batch"] * case["oc"] * oh * ow
    return {"bytes": 2 * (x + y * (1 + case["add"]) + case["oc"] * fan), "flops": 2 * y * fan}


def tolerance(case):
    """Whole numbers: every implementation of these operations gives the same bits."""
    return "exact"


# ------------------------------------------- the same in 64 bits, plain torch
def _sat(v):
    return v.clamp(-32768, 32767)


def _finish(acc, add, act):
    """32-bit wrap, the shift back to Q8.8, saturation, then the fused Add and activation."""
    v = _sat((((acc + (1 << 31)) & 0xFFFFFFFF) - (1 << 31)) >> 8)
    if add is not None:
        v = _sat(v + add)
    if act == "relu":
        v = v.clamp(min=0)
    elif act == "relu6":
        v = v.clamp(0, 1536)
    return v.to(torch.int16)


def _windows(x, c, oh, ow, kh, kw, s, p, d, fill):
    """One [..., oh, ow] view of x for each place of the window."""
    x = torch.nn.functional.pad(x, (p, p + d * kw + s, p, p + d * kh + s), value=fill)
    for i in range(kh):
        for j in range(kw):
            yield x[..., i * d:i * d + s * (oh - 1) + 1:s, j * d:j * d + s * (ow - 1) + 1:s]


def exact(case, seed):
    kind = case["kind"]
    if kind == "mobilenet":
        return None
    if kind == "mlp":
        x = _uniform(_gen(case, seed), case["batch"] * wl.MLP_IN, -1.0, 1.0).double().view(-1, wl.MLP_IN)
        for i, o, ids, act in ((wl.MLP_IN, wl.MLP_HIDDEN, (1, 2), "relu"), (wl.MLP_HIDDEN, wl.MLP_OUT, (3, 4), "none")):
            w = torch.from_numpy(wl.normal_q88(wl.rng(1, ids[0]), (i, o), 0.1)).to(DEV).double()
            b = torch.from_numpy(wl.normal_q88(wl.rng(1, ids[1]), (o,), 0.05)).to(DEV).long()
            x = _finish((x @ w).long(), b, act).double()
        return x.to(torch.int16).cpu().numpy()
    st = prepare(case, seed)
    if kind == "vectorop":
        a, b = st["a"].long().view(case["outer"], -1), st["b"].long()
        op = case["op"]
        if op == "div":
            q = torch.where(b == 0, 0, (a.abs() * 256) // b.abs().clamp(min=1))
            v = torch.where((a < 0) != (b < 0), -q, q)
        else:
            v = {"add": lambda: a + b, "sub": lambda: a - b, "mul": lambda: (a * b) >> 8,
                 "relu": lambda: a.clamp(min=0), "relu6": lambda: a.clamp(0, 1536)}[op]()
        return _sat(v).to(torch.int16).view(-1)
    if kind == "matmul":
        b, n, k, m = case["batch"], case["n"], case["k"], case["m"]
        acc = torch.stack([p @ q for p, q in zip(st["a"].double().view(b, n, k), st["b"].double().view(b, k, m))])
        add = None if st["add"] is None else st["add"].long().view((m,) if case["add"] == "column" else (b, n, m))
        return _finish(acc.long(), add, case["act"]).view(-1)
    if kind == "pool":
        if case["type"] != "max":      # the finalisers round in 32-bit floats by definition
            return None
        kh, kw, s, p, oh, ow = _pool_shape(case)
        x = st["x"].view(case["batch"], case["ch"], case["h"], case["w"])
        if case["k"] == 0:
            return x.amax((2, 3)).view(-1)
        v = None
        for t in _windows(x, case, oh, ow, kh, kw, s, p, 1, -32768):
            v = t if v is None else torch.maximum(v, t)
        return v.reshape(-1)
    oh, ow = _conv_out(case)
    y, w, k = [], st["w"].double(), case["k"]
    x = st["x"].view(case["batch"], case["ic"], case["h"], case["w"])
    add = None if st["add"] is None else st["add"].long().view(case["batch"], case["oc"], oh, ow)
    bias = (st["b"].long() << 8).view(-1, 1, 1)
    for i in range(case["batch"]):
        acc = torch.zeros(case["oc"], oh, ow, dtype=torch.float64, device=DEV)
        for t, v in enumerate(_windows(x[i].double(), case, oh, ow, k, k, case["stride"], case["pad"], case["dil"], 0.0)):
            if case["dw"]:
                acc += w.view(-1, k * k)[:, t].view(-1, 1, 1) * v
            else:
                acc += (w.view(case["oc"], case["ic"], k * k)[:, :, t].contiguous() @ v.reshape(case["ic"], -1)).view(-1, oh, ow)
        y.append(_finish(acc.long() + bias, None if add is None else add[i], case["act"]))
    return torch.stack(y).view(-1)

"""Performance cases of the tensor backend: the calls a user's program makes,
through the two public entry points (the C ABI of ``camel_amd._hip`` on device
buffers, the operators and layer chains of ``camel_amd.tensor``).

``listed()`` gives fixed cases, ``draw(rng)`` further ones of the same ranges,
``prepare(case, seed)`` the inputs, weights and output buffers a program holds
before the call, ``run(state)`` one pass, ``work(case)`` the bytes and
operations the pass cannot do without, ``exact(case, seed)`` the result in 64
bits and ``tolerance(case)`` how far a correct fp32 implementation may be off.
"""
from __future__ import annotations

import ctypes as C
import math

import torch
import torch.nn.functional as F

from camel_amd import _hip as H
from camel_amd import tensor as T

P = C.c_void_p
F32, F64 = torch.float32, torch.float64

MLP_IN, MLP_HIDDEN, MLP_CLASSES = 784, 1024, 10
MAX_GEMM = 4096 ** 3                      # multiply-adds of the largest matmul
MAX_CONV = 64 * 56 * 56 * 64 * 9 * 128    # and of the largest convolution
MAX_ELEMENTS = 1 << 28
ELTWISE = ("add", "subtract", "multiply", "scale", "relu", "relu_idiom")


def listed():
    return [
        # The smallest matmul of the benchmark set: launch latency counts.
        {"name": "matmul_256", "kind": "gemm", "M": 256, "N": 256, "K": 256, "trans": False,
         "bias": False, "relu": False},
        # The headline matmul.
        {"name": "matmul_4096", "kind": "gemm", "M": 4096, "N": 4096, "K": 4096, "trans": False,
         "bias": False, "relu": False},
        # A dense + bias + relu layer of a user's own sizes: nothing is a
        # multiple of a tile and the rows are not 16-byte aligned.
        {"name": "dense_ragged", "kind": "gemm", "M": 1000, "N": 3001, "K": 2047, "trans": False,
         "bias": True, "relu": True},
        # Backward of a dense layer, the weight gradient transpose(X) @ E over
        # a batch of 8192 rows.
        {"name": "dense_grad", "kind": "gemm", "M": 1024, "N": 1024, "K": 8192, "trans": True,
         "bias": False, "relu": False},
        # A dense layer applied to a few rows (serving): reading the weights
        # is the work.
        {"name": "dense_decode", "kind": "gemm", "M": 16, "N": 4096, "K": 4096, "trans": False,
         "bias": False, "relu": False},
        # MLP classifier forward as a composed layer chain, the benchmark's batch.
        {"name": "mlp_1024", "kind": "mlp", "batch": 1024, "hidden": MLP_HIDDEN, "layers": 2},
        # The benchmark's convolution layer.
        {"name": "conv_56", "kind": "conv", "N": 64, "C": 64, "H": 56, "W": 56, "Co": 128,
         "KS": 3, "stride": 1, "pad": 1},
        # A strided (downsampling) convolution of odd extents.
        {"name": "conv_strided", "kind": "conv", "N": 16, "C": 96, "H": 55, "W": 55, "Co": 160,
         "KS": 3, "stride": 2, "pad": 1},
        # Image classifier forward as a composed layer chain, the benchmark's batch.
        {"name": "cnn_512", "kind": "cnn", "batch": 512, "size": 28, "chans": 1},
        # One training step of a softmax regression at MNIST width: forward,
        # gradients, update, predictions; small operator calls.
        {"name": "train_step", "kind": "train", "rows": 1024, "features": 785, "classes": 10},
        # Elementwise at the benchmark's size: HBM bandwidth.
        {"name": "add_2e28", "kind": "eltwise", "op": "add", "n": MAX_ELEMENTS},
        # Row softmax at the benchmark's size.
        {"name": "softmax_1024", "kind": "softmax", "rows": 262144, "cols": 1024},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm; a third of them
    whole multiples of 64 where there is room for that."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 1 / 3:
        v -= v % 64
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "gemm", "mlp", "conv", "conv", "cnn", "train", "eltwise",
                       "softmax"))
    if kind == "gemm":
        while True:
            form = rng.choice(("square", "decode", "grad"))
            M = _log(rng, 1, 32) if form == "decode" else _log(rng, 64, 8192)
            N, K = _log(rng, 64, 8192), _log(rng, 64, 8192)
            if M * N * K <= MAX_GEMM:
                break
        epi = form != "grad" and rng.random() < 0.5
        return {"kind": kind, "M": M, "N": N, "K": K, "trans": form == "grad", "bias": epi,
                "relu": epi}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 1, 4096), "hidden": _log(rng, 64, 2048),
                "layers": rng.choice((1, 2, 3))}
    if kind == "conv":
        while True:
            hw = _log(rng, 7, 112)
            c = {"kind": kind, "N": _log(rng, 1, 64), "C": _log(rng, 1, 256), "H": hw,
                 "W": max(7, hw + rng.choice((0, 0, 0, 1, -3))), "Co": _log(rng, 16, 256),
                 "KS": rng.choice((1, 3, 3, 3, 5)), "stride": rng.choice((1, 1, 2))}
            c["pad"] = c["KS"] // 2
            oh, ow = _conv_out(c)
            if c["N"] * oh * ow * c["C"] * c["KS"] ** 2 * c["Co"] <= MAX_CONV:
                return c
    if kind == "cnn":
        return {"kind": kind, "batch": _log(rng, 1, 512), "size": rng.choice((20, 28, 32)),
                "chans": rng.choice((1, 1, 3))}
    if kind == "train":
        return {"kind": kind, "rows": _log(rng, 100, 16384), "features": _log(rng, 33, 1024),
                "classes": rng.choice((2, 10, 10, 26, 100))}
    if kind == "eltwise":
        return {"kind": kind, "op": rng.choice(ELTWISE), "n": _log(rng, 1 << 10, MAX_ELEMENTS)}
    while True:
        c = {"kind": kind, "rows": _log(rng, 16, 262144), "cols": _log(rng, 2, 32768)}
        if c["rows"] * c["cols"] <= MAX_ELEMENTS:
            return c


# ---- inputs ------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(g, *shape, lo=-1.0, hi=1.0):
    return torch.rand(*shape, generator=g, device="cuda", dtype=F32) * (hi - lo) + lo


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=F32) * std


def _conv_out(c):
    return ((c["H"] + 2 * c["pad"] - c["KS"]) // c["stride"] + 1,
            (c["W"] + 2 * c["pad"] - c["KS"]) // c["stride"] + 1)


def _mlp_dims(case):
    return [MLP_IN] + [case["hidden"]] * case["layers"] + [MLP_CLASSES]


def _cnn_flat(case):
    return 64 * ((case["size"] - 4) // 2) ** 2


def _inputs(case, seed):
    """The case's input tensors (torch, on the GPU), by name."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        v = {"A": _uniform(g, *((K, M) if case["trans"] else (M, K))), "B": _uniform(g, K, N)}
        if case["bias"]:
            v["bias"] = _uniform(g, N)
        return v
    if kind == "mlp":
        d = _mlp_dims(case)
        v = {"x": _uniform(g, case["batch"], d[0], lo=0.0)}
        for i in range(len(d) - 1):
            v[f"w{i}"] = _normal(g, d[i], d[i + 1], std=d[i] ** -0.5)
            v[f"b{i}"] = _uniform(g, d[i + 1], lo=-0.1, hi=0.1)
        return v
    if kind == "conv":
        k = case["C"] * case["KS"] ** 2
        return {"x": _normal(g, case["N"], case["C"], case["H"], case["W"]),
                "w": _normal(g, case["Co"], case["C"], case["KS"], case["KS"], std=(2.0 / k) ** 0.5),
                "b": _uniform(g, case["Co"], lo=-0.1, hi=0.1)}
    if kind == "cnn":
        ch, flat = case["chans"], _cnn_flat(case)
        return {"x": _uniform(g, case["batch"], ch, case["size"], case["size"], lo=0.0),
                "w1": _normal(g, 32, ch, 3, 3, std=(2.0 / (9 * ch)) ** 0.5),
                "b1": _uniform(g, 32, lo=-0.1, hi=0.1),
                "w2": _normal(g, 64, 32, 3, 3, std=(2.0 / 288) ** 0.5),
                "b2": _uniform(g, 64, lo=-0.1, hi=0.1),
                "w3": _normal(g, flat, 128, std=(2.0 / flat) ** 0.5),
                "b3": _uniform(g, 128, lo=-0.1, hi=0.1),
                "w4": _normal(g, 128, 10, std=(2.0 / 128) ** 0.5),
                "b4": _uniform(g, 10, lo=-0.1, hi=0.1)}
    if kind == "train":
        n, d, k = case["rows"], case["features"], case["classes"]
        label = torch.randint(0, k, (n,), generator=g, device="cuda")
        return {"X": _uniform(g, n, d, lo=0.0), "Y": F.one_hot(label, k).to(F32),
                "W": _normal(g, d, k, std=d ** -0.5), "b": _uniform(g, k, lo=-0.1, hi=0.1)}
    if kind == "eltwise":
        v = {"l": _normal(g, case["n"])}
        if case["op"] in ("add", "subtract", "multiply"):
            v["r"] = _normal(g, case["n"])
        return v
    return {"x": _normal(g, case["rows"], case["cols"], std=2.0)}


class _Result:
    """A tensor of the operator layer seen by torch without a copy; the handle
    is released with the last view."""

    def __init__(self, t):
        code, shape = t.meta()
        self.t = t
        self.__cuda_array_interface__ = {
            "shape": shape, "typestr": {T.TC_FLOAT32: "<f4", T.TC_INT64: "<i8"}[code],
            "data": (t.device_ptr(), False), "version": 2}

    def __del__(self):
        self.t.release()


def _seen(t):
    return torch.as_tensor(_Result(t), device="cuda")


def _empty(*shape, dtype=F32):
    return torch.empty(*shape, device="cuda", dtype=dtype)


class _State:
    """Inputs, weights and handles a program holds before the call."""

    def __init__(self, case):
        self.case = case
        self.chain, self.handles = None, {}

    def __del__(self):
        if self.chain is not None:
            self.chain.release()
        for t in self.handles.values():
            t.release()


def prepare(case, seed):
    s = _State(case)
    kind = case["kind"]
    v = _inputs(case, seed)
    if kind in ("mlp", "cnn", "train"):
        # Operator-layer programs hold tensors of the layer.
        torch.cuda.synchronize()
        s.handles = {k: T.Tensor.from_dlpack(x.contiguous()) for k, x in v.items()}
        h = s.handles
        if kind == "mlp":
            last = len(_mlp_dims(case)) - 2
            layers = []
            for i in range(last + 1):
                layers.append(("dense", h[f"w{i}"], h[f"b{i}"]))
                layers.append("relu" if i < last else "softmax")
            s.chain = T.Chain(*layers)
        elif kind == "cnn":
            s.chain = T.Chain(("conv2d", h["w1"], h["b1"]), "relu",
                              ("conv2d", h["w2"], h["b2"]), "relu", ("maxpool2d", 2, 2),
                              ("reshape", case["batch"], _cnn_flat(case)),
                              ("dense", h["w3"], h["b3"]), "relu",
                              ("dense", h["w4"], h["b4"]), "softmax")
        return s
    # Programs on the C ABI hold device buffers, the result's among them.
    s.v = v
    if kind == "gemm":
        s.out = _empty(case["M"], case["N"])
        s.flags = ((H.EPI_BIAS if case["bias"] else 0) | (H.EPI_RELU if case["relu"] else 0) |
                   (H.GEMM_A_T if case["trans"] else 0))
    elif kind == "conv":
        s.out = _empty(case["N"], case["Co"], *_conv_out(case))
    elif kind == "eltwise":
        s.out = _empty(case["n"])
        if case["op"] == "relu_idiom":
            s.mask = _empty(case["n"], dtype=torch.uint8)
    else:
        s.out = _empty(case["rows"], case["cols"])
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------

def _ptr(t):
    return P(t.data_ptr())


def _run_train(s):
    # The update step of a softmax regression (mnist.cml's, with a bias).
    h, n = s.handles, s.case["rows"]
    logits = T.call("dense", h["X"], with_=(h["W"], h["b"]))
    probs = T.call("softmax", logits)
    err = T.call("subtract", probs, h["Y"])
    xt = T.call("transpose", h["X"])
    grad = T.call("matmul", xt, err)
    gbias = T.call("sum_axis", err, 0)
    rate = 0.1 / n
    step = T.call("multiply", rate, grad)
    w = T.call("subtract", h["W"], step)
    bstep = T.call("multiply", rate, gbias)
    b = T.call("subtract", h["b"], bstep)
    pred = T.call("argmax_axis", probs, 1)
    for t in (err, xt, step, bstep):
        t.release()
    return {"logits": _seen(logits), "probs": _seen(probs), "grad": _seen(grad),
            "gbias": _seen(gbias), "w": _seen(w), "b": _seen(b), "pred": _seen(pred)}


def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "gemm":
        H.call("camel_hip_sgemm", _ptr(s.v["A"]), _ptr(s.v["B"]), _ptr(s.out), c["M"], c["N"],
               c["K"], _ptr(s.v["bias"]) if c["bias"] else None, s.flags)
    elif kind in ("mlp", "cnn"):
        return _seen(s.chain(s.handles["x"]))
    elif kind == "conv":
        H.call("camel_hip_conv2d", _ptr(s.v["x"]), _ptr(s.v["w"]), _ptr(s.v["b"]), _ptr(s.out),
               c["N"], c["C"], c["H"], c["W"], c["Co"], c["KS"], c["KS"], c["stride"], c["pad"],
               H.EPI_BIAS | H.EPI_RELU)
    elif kind == "train":
        return _run_train(s)
    elif kind == "softmax":
        H.call("camel_hip_softmax_rows", _ptr(s.v["x"]), _ptr(s.out), c["rows"], c["cols"])
    else:
        op, n, l = c["op"], c["n"], _ptr(s.v["l"])
        if op == "relu":
            H.call("camel_hip_relu", l, _ptr(s.out), n)
        elif op == "scale":
            H.call("camel_hip_binary_scalar", H.OP_MUL, 0, H.DT_F32, l, 0.37, H.DT_F32,
                   _ptr(s.out), n)
        elif op == "relu_idiom":
            # multiply(x, x > 0): a Bool tensor, then a mixed-type product.
            H.call("camel_hip_compare_scalar", H.CMP_GT, 0, H.DT_F32, l, 0.0, _ptr(s.mask), n)
            H.call("camel_hip_binary", H.OP_MUL, H.DT_F32, l, H.DT_BOOL, _ptr(s.mask), H.DT_F32,
                   _ptr(s.out), n)
            return s.out, s.mask
        else:
            code = {"add": H.OP_ADD, "subtract": H.OP_SUB, "multiply": H.OP_MUL}[op]
            H.call("camel_hip_binary", code, H.DT_F32, l, H.DT_F32, _ptr(s.v["r"]), H.DT_F32,
                   _ptr(s.out), n)
    return s.out


# ---- what a pass cannot do without ---------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if kind == "mlp":
        d, n = _mlp_dims(case), case["batch"]
        macs = sum(d[i] * d[i + 1] for i in range(len(d) - 1))
        return {"bytes": 4 * (n * (d[0] + d[-1]) + macs + sum(d[1:])), "flops": 2 * n * macs}
    if kind == "conv":
        oh, ow = _conv_out(case)
        wn = case["Co"] * case["C"] * case["KS"] ** 2
        out = case["N"] * oh * ow
        return {"bytes": 4 * (case["N"] * case["C"] * case["H"] * case["W"] + wn +
                              out * case["Co"]),
                "flops": 2 * out * wn}
    if kind == "cnn":
        n, ch, s, flat = case["batch"], case["chans"], case["size"], _cnn_flat(case)
        macs = ((s - 2) ** 2 * 32 * 9 * ch + (s - 4) ** 2 * 64 * 288 + flat * 128 + 1280)
        return {"bytes": 4 * (n * (ch * s * s + 10) + 288 * ch + 64 * 288 + flat * 128 + 1280),
                "flops": 2 * n * macs}
    if kind == "train":
        n, d, k = case["rows"], case["features"], case["classes"]
        return {"bytes": 4 * (n * d + n * k * 3 + 3 * d * k) + 8 * n, "flops": 4 * n * d * k}
    if kind == "eltwise":
        per = {"add": 12, "subtract": 12, "multiply": 12, "scale": 8, "relu": 8,
               "relu_idiom": 9}[case["op"]]
        return {"bytes": per * case["n"], "flops": case["n"]}
    n = case["rows"] * case["cols"]
    return {"bytes": 8 * n, "flops": 4 * n}


# ---- results in 64 bits ----------------------------------------------------------

def _relu(x):
    return x.clamp_min(0)


def _conv64(x, w, b, stride, pad):
    """im2col in float64, a few images at a time."""
    n, c, hh, ww = x.shape
    co, ks = w.shape[0], w.shape[2]
    oh, ow = (hh + 2 * pad - ks) // stride + 1, (ww + 2 * pad - ks) // stride + 1
    out = torch.empty(n, co, oh, ow, device=x.device, dtype=F64)
    w2 = w.reshape(co, -1).to(F64)
    for i in range(n):
        cols = F.unfold(x[i:i + 1].to(F64), ks, padding=pad, stride=stride)[0]
        out[i] = (w2 @ cols + b.to(F64)[:, None]).reshape(co, oh, ow)
    return out


def exact(case, seed):
    v = _inputs(case, seed)
    kind = case["kind"]
    if kind == "gemm":
        a = v["A"].to(F64)
        y = (a.t().contiguous() if case["trans"] else a) @ v["B"].to(F64)
        if case["bias"]:
            y += v["bias"].to(F64)
        return _relu(y) if case["relu"] else y
    if kind == "mlp":
        h = v["x"].to(F64)
        last = len(_mlp_dims(case)) - 2
        for i in range(last + 1):
            h = h @ v[f"w{i}"].to(F64) + v[f"b{i}"].to(F64)
            h = _relu(h) if i < last else torch.softmax(h, 1)
        return h
    if kind == "conv":
        return _relu(_conv64(v["x"], v["w"], v["b"], case["stride"], case["pad"]))
    if kind == "cnn":
        h = _relu(_conv64(v["x"], v["w1"], v["b1"], 1, 0))
        h = _relu(_conv64(h, v["w2"], v["b2"], 1, 0))
        h = F.max_pool2d(h, 2).reshape(case["batch"], -1)
        h = _relu(h @ v["w3"].to(F64) + v["b3"].to(F64))
        return torch.softmax(h @ v["w4"].to(F64) + v["b4"].to(F64), 1)
    if kind == "train":
        X, Y, W, b = (v[k].to(F64) for k in ("X", "Y", "W", "b"))
        logits = X @ W + b
        probs = torch.softmax(logits, 1)
        err = probs - Y
        grad, gbias = X.t().contiguous() @ err, err.sum(0)
        rate = 0.1 / case["rows"]
        return {"logits": logits, "probs": probs, "grad": grad, "gbias": gbias,
                "w": W - rate * grad, "b": b - rate * gbias, "pred": probs.argmax(1)}
    if kind == "eltwise":
        l, op = v["l"].to(F64), case["op"]
        if op == "relu":
            return l * (l > 0)
        if op == "relu_idiom":
            mask = l > 0
            return l * mask, mask.to(torch.uint8)
        if op == "scale":
            return l * 0.37
        r = v["r"].to(F64)
        return l + r if op == "add" else l - r if op == "subtract" else l * r
    return torch.softmax(v["x"].to(F64), 1)


def tolerance(case):
    # About four times the largest error against 64 bits that was measured
    # over these ranges (matmul 1.1e-6 at K = 4096 and 8192, MLP and CNN
    # probabilities 3e-7, training step 9e-8, softmax 4e-8); two correct
    # summation orders differ by no more.
    kind = case["kind"]
    if kind == "eltwise":
        return "exact"  # one IEEE operation per element
    if kind == "softmax":
        return {"rel": 2e-7, "max": 2e-6}
    if kind == "train":
        return {"rel": 1e-6, "max": 4e-5, "differ": 2e-3}
    if kind in ("mlp", "cnn"):
        return {"rel": 2e-6, "max": 8e-5}
    return {"rel": 5e-6, "max": 1e-4}

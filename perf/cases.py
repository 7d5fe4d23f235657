"""The workloads whose speed this repository follows: fp32 GEMM, batched GEMM,
Linear and Conv2D, forward and backward, through the package's public calls.

Sizes are those of bench.py and the tests (the square and small products, the
transposed and sliced views, the fully connected layer, the 3x3 and 1x1
convolution layers and the 7x7 stem at batch 32) or generic ragged ones.
Every state holds what a training or inference program holds before the call:
inputs, weights, the incoming gradient, and the output it accumulates into;
outputs and scratch memory are left to the call.
"""
import math

import torch
import torch.nn.functional as F

import minitensor_amd as mt

DEV = "cuda"


def listed():
    return [
        # the smallest product of the benchmark: a call's fixed cost shows
        dict(name="matmul_small", kind="gemm", m=256, n=512, k=512, ta=False, tb=False,
             skip=0, bias="none", beta=0.0),
        # the headline product: a compute-bound square GEMM, and the largest work
        dict(name="matmul_large", kind="gemm", m=4096, n=4096, k=4096, ta=False, tb=False,
             skip=0, bias="none", beta=0.0),
        # a row slice times a transposed view, read in place (attention scores, x·wᵀ)
        dict(name="view_slice", kind="gemm", m=1920, n=2048, k=1024, ta=False, tb=True,
             skip=128, bias="none", beta=0.0),
        # ragged sizes (rows not 16-byte aligned), bias, accumulation into C
        dict(name="ragged_bias_beta", kind="gemm", m=1027, n=1285, k=771, ta=False, tb=False,
             skip=0, bias="col", beta=0.5),
        # one row against a square weight: a single sample, bound by the weight's bytes
        dict(name="matvec", kind="gemm", m=1, n=4096, k=4096, ta=False, tb=False,
             skip=0, bias="none", beta=0.0),
        # attention-like batch of short-K products, output-bound
        dict(name="bmm", kind="bmm", b=64, m=512, n=512, k=64),
        # a classifier head's training step: forward, dX, dW, db
        dict(name="linear_train", kind="linear", rows=256, fin=2048, fout=1000, beta=0.0),
        # a small MLP layer's training step, gradients accumulated
        dict(name="linear_small_train", kind="linear", rows=64, fin=784, fout=130, beta=1.0),
        # a residual network's 3x3 layer: inference, then its backward
        dict(name="conv3x3_forward", kind="conv", n=32, c=256, h=14, w=14, co=256, k=3,
             stride=1, pad=1, forward=True, backward=False, dx=False),
        dict(name="conv3x3_backward", kind="conv", n=32, c=256, h=14, w=14, co=256, k=3,
             stride=1, pad=1, forward=False, backward=True, dx=True),
        # a downsampling 1x1 shortcut's training step
        dict(name="conv1x1_s2_train", kind="conv", n=32, c=256, h=56, w=56, co=512, k=1,
             stride=2, pad=0, forward=True, backward=True, dx=True),
        # the RGB stem's training step: the first layer needs no dX
        dict(name="stem_train", kind="conv", n=32, c=3, h=224, w=224, co=64, k=7,
             stride=2, pad=3, forward=True, backward=True, dx=False),
    ]


def _log_int(rng, lo, hi, aligned):
    """An integer spread over [lo, hi] by its logarithm; a multiple of 16
    above 32 when `aligned`."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if aligned and v > 32:
        v = max(lo, v // 16 * 16)
    return min(max(v, lo), hi)


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "bmm", "linear", "conv", "conv"])
    al = rng.random() < 0.6          # most programs' sizes are multiples of 16
    while True:
        if kind == "gemm":
            c = dict(kind="gemm", m=_log_int(rng, 1, 4096, al), n=_log_int(rng, 16, 4096, al),
                     k=_log_int(rng, 16, 4096, al), ta=rng.random() < 0.25,
                     tb=rng.random() < 0.4, skip=0, bias=rng.choice(["none", "none", "row", "col"]),
                     beta=rng.choice([0.0, 0.0, 0.5]))
            c["skip"] = rng.choice([0, 0, 128]) if not c["ta"] else 0
            cap = 4e10
        elif kind == "bmm":
            c = dict(kind="bmm", b=_log_int(rng, 2, 128, False), m=_log_int(rng, 16, 512, al),
                     n=_log_int(rng, 16, 512, al), k=_log_int(rng, 16, 256, al))
            cap = 8e9
        elif kind == "linear":
            c = dict(kind="linear", rows=_log_int(rng, 8, 4096, al), fin=_log_int(rng, 64, 4096, al),
                     fout=_log_int(rng, 10, 4096, al), beta=rng.choice([0.0, 1.0]))
            cap = 2e10
        else:
            k = rng.choice([1, 1, 3, 3, 3, 5])
            hw = rng.choice([7, 13, 14, 28, 32, 56])
            stride = rng.choice([1, 1, 2])
            fwd = rng.random() < 0.6
            c = dict(kind="conv", n=_log_int(rng, 1, 32, False), c=_log_int(rng, 3, 512, al), h=hw,
                     w=hw, co=_log_int(rng, 16, 512, al), k=k, stride=stride, pad=k // 2,
                     forward=fwd, backward=not fwd or rng.random() < 0.5, dx=True)
            cap = 1e10
        w = work(c)
        if w["flops"] <= cap and w["bytes"] <= 4e8:
            return c


def _out_hw(c):
    o = lambda v: (v + 2 * c["pad"] - c["k"]) // c["stride"] + 1  # noqa: E731
    return o(c["h"]), o(c["w"])


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, device=DEV, generator=g) * 2 - 1


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g) * std


def prepare(case, seed):
    g = _generator(seed)
    s = dict(case=case)
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s["a"] = _uniform(g, k, m).t() if case["ta"] else _uniform(g, case["skip"] + m, k)[case["skip"]:]
        s["b"] = _uniform(g, n, k).t() if case["tb"] else _uniform(g, k, n)
        s["bias"] = None
        if case["bias"] != "none":
            s["bias"] = _normal(g, m if case["bias"] == "row" else n, std=0.1)
        s["axis"] = {"none": mt.BIAS_NONE, "row": mt.BIAS_ROW, "col": mt.BIAS_COL}[case["bias"]]
        s["c"] = _uniform(g, m, n) if case["beta"] else None
    elif case["kind"] == "bmm":
        s["a"] = _uniform(g, case["b"], case["m"], case["k"])
        s["b"] = _uniform(g, case["b"], case["k"], case["n"])
    elif case["kind"] == "linear":
        r, fi, fo = case["rows"], case["fin"], case["fout"]
        # activations after a ReLU, He weights, a loss gradient's scale
        s["x"] = torch.relu(_normal(g, r, fi))
        s["w"] = _normal(g, fo, fi, std=(2.0 / fi) ** 0.5)
        s["bias"] = _normal(g, fo, std=0.1)
        s["dy"] = _normal(g, r, fo, std=0.01)
        s["dw"] = _normal(g, fo, fi, std=0.01) if case["beta"] else None
        s["db"] = _normal(g, fo, std=0.01) if case["beta"] else None
    else:
        n, c, h, w, co, k = (case[x] for x in ("n", "c", "h", "w", "co", "k"))
        ho, wo = _out_hw(case)
        x = _normal(g, n, c, h, w)
        s["x"] = x if c == 3 else torch.relu(x)   # an image, or a hidden activation
        s["w"] = _normal(g, co, c, k, k, std=(2.0 / (c * k * k)) ** 0.5)
        s["bias"] = _normal(g, co, std=0.1)
        s["dy"] = _normal(g, n, co, ho, wo, std=0.01) if case["backward"] else None
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "gemm":
        if s["bias"] is None and s["c"] is None:
            return mt.matmul(s["a"], s["b"])
        return mt.gemm(s["a"], s["b"], out=s["c"], bias=s["bias"], bias_axis=s["axis"],
                       beta=case["beta"])
    if case["kind"] == "bmm":
        return mt.bmm(s["a"], s["b"])
    if case["kind"] == "linear":
        y = mt.linear(s["x"], s["w"], s["bias"])
        dx, dw, db = mt.linear_backward(s["dy"], s["x"], s["w"], dw=s["dw"], db=s["db"],
                                        beta_w=case["beta"], beta_b=case["beta"])
        return {"y": y, "dx": dx, "dw": dw, "db": db}
    out = {}
    if case["forward"]:
        out["y"] = mt.conv2d(s["x"], s["w"], s["bias"], case["stride"], case["pad"])
    if case["backward"]:
        dx, dw, db = mt.conv2d_backward(s["x"], s["w"], s["dy"], case["stride"], case["pad"],
                                        need_dx=case["dx"])
        out["dw"], out["db"] = dw, db
        if case["dx"]:
            out["dx"] = dx
    return out


def work(case):
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        b = m * k + k * n + m * n * (2 if case["beta"] else 1)
        b += {"none": 0, "row": m, "col": n}[case["bias"]]
        return {"bytes": 4 * b, "flops": 2 * m * n * k}
    if case["kind"] == "bmm":
        b, m, n, k = case["b"], case["m"], case["n"], case["k"]
        return {"bytes": 4 * b * (m * k + k * n + m * n), "flops": 2 * b * m * n * k}
    if case["kind"] == "linear":
        r, fi, fo = case["rows"], case["fin"], case["fout"]
        # x, w, dy and the bias read; y, dx, dw, db written (dw, db also read to accumulate)
        grads = fo * fi + fo
        b = r * fi + fo * fi + fo + r * fo + r * fo + r * fi + grads * (2 if case["beta"] else 1)
        return {"bytes": 4 * b, "flops": 3 * 2 * r * fi * fo + r * fo}
    n, c, co, k = case["n"], case["c"], case["co"], case["k"]
    ho, wo = _out_hw(case)
    x, w, y = n * c * case["h"] * case["w"], co * c * k * k, n * co * ho * wo
    product = 2 * n * ho * wo * co * c * k * k
    b = x + w
    flops = 0
    if case["forward"]:
        b += co + y
        flops += product
    if case["backward"]:
        b += y + w + co + (x if case["dx"] else 0)
        flops += product * (2 if case["dx"] else 1) + y
    return {"bytes": 4 * b, "flops": flops}


def tolerance(case):
    # 32-bit products and sums: measured against 64 bits, the outputs are 7e-8
    # to 1.1e-6 off in the 2-norm (the longest sums, K = 4096, the most), single
    # elements up to 1.1e-5 of the rms; two implementations differ by both.
    return {"rel": 5e-6, "max": 1e-4}


def _conv_columns(x, case):
    return F.unfold(x[None], case["k"], padding=case["pad"], stride=case["stride"])[0]


def exact(case, seed):
    s = prepare(case, seed)
    d = {k: v.double() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if case["kind"] == "gemm":
        r = d["a"] @ d["b"]
        if case["bias"] == "row":
            r += d["bias"][:, None]
        elif case["bias"] == "col":
            r += d["bias"][None, :]
        if case["beta"]:
            r += case["beta"] * d["c"]
        return r
    if case["kind"] == "bmm":
        return torch.stack([a @ b for a, b in zip(d["a"], d["b"])])
    if case["kind"] == "linear":
        dw, db = d["dy"].t() @ d["x"], d["dy"].sum(0)
        if case["beta"]:
            dw, db = dw + case["beta"] * d["dw"], db + case["beta"] * d["db"]
        return {"y": d["x"] @ d["w"].t() + d["bias"], "dx": d["dy"] @ d["w"], "dw": dw, "db": db}
    n, co = case["n"], case["co"]
    ho, wo = _out_hw(case)
    wm = d["w"].reshape(co, -1)
    y, dx, dw = [], [], torch.zeros_like(wm)
    for i in range(n):
        col = _conv_columns(d["x"][i], case)
        if case["forward"]:
            y.append((wm @ col + d["bias"][:, None]).reshape(co, ho, wo))
        if case["backward"]:
            dy = d["dy"][i].reshape(co, -1)
            dw += dy @ col.t()
            if case["dx"]:
                dx.append(F.fold((wm.t() @ dy)[None], (case["h"], case["w"]), case["k"],
                                 padding=case["pad"], stride=case["stride"])[0])
    out = {}
    if case["forward"]:
        out["y"] = torch.stack(y)
    if case["backward"]:
        out["dw"], out["db"] = dw.reshape(d["w"].shape), d["dy"].sum((0, 2, 3))
        if case["dx"]:
            out["dx"] = torch.stack(dx)
    return out

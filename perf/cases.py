"""What this library's speed is measured on: the work its users have it do, through the public entry points, over the
range of sizes that its benchmark, tests and examples span.

Seven kinds of work:
  gemm          one fp16-rounded product of two matrices (nz::data::iTensorCoreGEMM on single matrices)
  linear        forward of a fully connected layer in serving: fused bias and ReLU, optionally with the weights' fp16 image
                kept in a handle, as nz::Model keeps it while the weights do not change
  linear_train  one training step of such a layer inside a network: forward with ReLU, its bias, weight and data gradients for the
                output gradient that comes from above, SGD
  batched       a 4-D batch of products (multi-head shaped)
  conv          forward of a Conv2d layer in serving, shared weights with a per-channel bias or the reference's own
                parameters (one weight copy per image, a bias per pixel and channel)
  conv_train    forward and all gradients of a Conv2d + ReLU layer with the reference's per-pixel bias
  readme_step   one Adam training step of the reference's README network (README.md:62-90)

Operands are fp32 in memory, rounded to fp16 by the library and accumulated in fp32: there is no other data type on
this path.
"""
from __future__ import annotations

import math

import torch

from neuzephyr_amd import capi

# The largest drawn product does the work of the largest listed one at most; convolutions and batches, which run further
# from the matrix pipes' rate, are kept to an eighth of its multiplications.
MAX_FLOPS = 2.0 * 8192 ** 3


def listed():
    return [
        # a small dense product, where the launch and the latency of one pass over k count
        {"name": "gemm_256", "kind": "gemm", "M": 256, "K": 256, "N": 256, "b_trans": False},
        # odd extents in all three directions: rows that allow no 16-byte loads
        {"name": "gemm_ragged", "kind": "gemm", "M": 1000, "K": 777, "N": 513, "b_trans": False},
        # the headline product
        {"name": "gemm_8192", "kind": "gemm", "M": 8192, "K": 8192, "N": 8192, "b_trans": False},
        # one sample through a layer: the weights are streamed once
        {"name": "linear_one_sample", "kind": "linear", "samples": 1, "inputs": 4096, "outputs": 4096, "kept": False},
        # a batch through a layer in serving
        {"name": "linear_batch", "kind": "linear", "samples": 4096, "inputs": 1024, "outputs": 4096, "kept": True},
        # the same layer in training
        {"name": "linear_train", "kind": "linear_train", "samples": 4096, "inputs": 1024, "outputs": 4096},
        # attention-shaped batch of products
        {"name": "batched", "kind": "batched", "n": 8, "c": 16, "M": 1024, "K": 1024, "N": 1024},
        # a wide 3x3 layer in serving
        {"name": "conv_wide", "kind": "conv", "n": 16, "C": 64, "H": 128, "W": 128, "O": 128, "K": 3, "stride": 1, "pad": 1,
         "per_sample": False, "kept": True},
        # the memory-bound layer: three channels into one
        {"name": "conv_thin", "kind": "conv", "n": 10, "C": 3, "H": 1024, "W": 1024, "O": 1, "K": 3, "stride": 1, "pad": 1,
         "per_sample": False, "kept": False},
        # a deep layer on 14 x 14 images in training, one set of weights for all images
        {"name": "conv_train_deep", "kind": "conv_train", "n": 16, "C": 256, "H": 14, "W": 14, "O": 256, "K": 3, "stride": 1,
         "pad": 1, "per_sample": False},
        # a down-sampling layer in training, in the reference's own parameter form
        {"name": "conv_train_strided", "kind": "conv_train", "n": 16, "C": 128, "H": 56, "W": 56, "O": 128, "K": 3, "stride": 2,
         "pad": 1, "per_sample": True},
        # the reference's example program
        {"name": "readme_step", "kind": "readme_step", "n": 10, "H": 1024, "W": 1024},
    ]


def _log(rng, lo, hi):
    """An extent spread over the logarithm of [lo, hi]; half of them as they fall (odd ones among them), half multiples of 16."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return v if rng.random() < 0.5 or v < 16 else v // 16 * 16


def _draw_conv(rng):
    """A layer of the shapes that image networks have: few channels on large images, many on small ones."""
    K, stride = rng.choice(((3, 1), (3, 1), (3, 1), (1, 1), (1, 1), (5, 1), (3, 2), (1, 2), (7, 2)))
    return {"n": rng.choice((1, 2, 4, 8, 10, 16, 16, 32)), "C": _log(rng, 3, 512), "H": _log(rng, 7, 224), "W": 0, "O": _log(rng, 8, 512),
            "K": K, "stride": stride, "pad": K // 2, "per_sample": rng.random() < 0.4}


def draw(rng):
    kind = rng.choice(("gemm", "linear", "linear_train", "batched", "conv", "conv", "conv_train", "conv_train", "readme_step"))
    while True:
        limit = MAX_FLOPS / 8
        if kind == "gemm":
            case = {"M": _log(rng, 64, 8192), "K": _log(rng, 64, 8192), "N": _log(rng, 64, 8192), "b_trans": rng.random() < 0.5}
            limit = MAX_FLOPS / 2
        elif kind == "linear":
            case = {"samples": _log(rng, 1, 4096), "inputs": _log(rng, 256, 8192), "outputs": _log(rng, 256, 8192),
                    "kept": rng.random() < 0.5}
        elif kind == "linear_train":
            case = {"samples": _log(rng, 16, 4096), "inputs": _log(rng, 256, 4096), "outputs": _log(rng, 256, 4096)}
        elif kind == "batched":
            case = {"n": rng.choice((1, 2, 4, 8)), "c": rng.choice((1, 4, 8, 12, 16)), "M": _log(rng, 64, 1024),
                    "K": _log(rng, 64, 1024), "N": _log(rng, 64, 1024)}
        elif kind == "readme_step":
            case = {"n": rng.choice((2, 4, 8, 10)), "H": rng.randrange(256, 1025), "W": rng.randrange(256, 1025)}
            if rng.random() < 0.5:                                          # half of the images have aligned rows
                case["W"] = case["W"] // 8 * 8
        else:
            case = _draw_conv(rng)
            case["W"] = case["H"] if rng.random() < 0.8 else _log(rng, 7, 224)
            if kind == "conv":
                case["kept"] = rng.random() < 0.5
                if rng.random() < 0.15:                                     # thin layers on large images
                    case.update(n=rng.choice((4, 8, 10)), C=rng.choice((1, 3)), O=rng.choice((1, 2)), K=3, stride=1, pad=1,
                                H=rng.randrange(256, 1025), W=rng.randrange(256, 1025) // 4 * 4)
            if min(case["H"], case["W"]) + 2 * case["pad"] < case["K"]:
                continue
            limit = MAX_FLOPS / 16
        case["kind"] = kind
        w = work(case)
        if w["flops"] <= limit and w["bytes"] <= 8.0e8:
            return case


def _outputs(case):
    K, s, p = case["K"], case["stride"], case["pad"]
    return (case["H"] + 2 * p - K) // s + 1, (case["W"] + 2 * p - K) // s + 1


def _readme_sizes(case):
    H, W = case["H"], case["W"]
    return (H - 5) // 2 + 1, (W - 5) // 2 + 1                               # 5 x 5 average pooling, stride 2, of same-size convolutions


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 4.0 * (M * K + K * N + M * N), "flops": 2.0 * M * K * N}
    if kind in ("linear", "linear_train"):
        S, I, O = case["samples"], case["inputs"], case["outputs"]
        if kind == "linear":
            return {"bytes": 4.0 * (S * I + I * O + O + S * O), "flops": 2.0 * S * I * O}
        # x, dy, W, b in; y, dx, dW, db, updated W and b out
        return {"bytes": 4.0 * (2 * S * I + 3 * I * O + 3 * O + 2 * S * O), "flops": 6.0 * S * I * O}
    if kind == "batched":
        b, M, K, N = case["n"] * case["c"], case["M"], case["K"], case["N"]
        return {"bytes": 4.0 * b * (M * K + K * N + M * N), "flops": 2.0 * b * M * K * N}
    if kind in ("conv", "conv_train"):
        Ho, Wo = _outputs(case)
        n, C, O, K = case["n"], case["C"], case["O"], case["K"]
        x, y = n * C * case["H"] * case["W"], n * O * Ho * Wo
        w = (n if case["per_sample"] else 1) * C * K * K * O
        b = Ho * Wo * O if case["per_sample"] or kind == "conv_train" else O
        flops = 2.0 * y * C * K * K
        if kind == "conv":
            return {"bytes": 4.0 * (x + w + b + y), "flops": flops}
        return {"bytes": 4.0 * (2 * x + 2 * w + 2 * b + 2 * y), "flops": 3 * flops}     # y and dy; x, dx, w, dw, b, db
    n, H, W = case["n"], case["H"], case["W"]
    hp, wp = _readme_sizes(case)
    # the input, the two convolutions' per-pixel biases and the linear weights with their gradients and Adam moments
    params = 2 * H * W + 16 * hp * wp
    flops = 2.0 * n * H * W * (27 * 2 + 9 * 3) + 2.0 * n * hp * wp * (25 * 2 + 16 * 3)
    return {"bytes": 4.0 * (3 * n * H * W + params * 7), "flops": flops}


def tolerance(case):
    kind = case["kind"]
    # The products are exact in fp32 and only the order of the fp32 sums is free: against 64-bit sums of the same rounded
    # operands the outputs of all kinds are off by 0.6e-7 to 6e-7 in the 2-norm and by 0.3e-6 to 4e-6 at worst.
    tol = {"rel": 2.5e-6, "max": 2e-5}
    if kind in ("linear_train", "conv_train"):
        # An activation that is zero up to rounding passes its gradient on or not, depending on the order of the forward's sums:
        # about one in five million (normal activations, sums good to 1.5e-7). Where one is likely, a gradient may have one
        # element of the output gradient more or less: 1 / sqrt(half of them) of its norm.
        y = case["samples"] * case["outputs"] if kind == "linear_train" else case["n"] * case["O"] * math.prod(_outputs(case))
        if y > 100_000:
            tol = {"rel": 3.0 / math.sqrt(y / 2), "max": 0.9}
    elif kind == "readme_step":
        # The softmax's and the loss's gradients (160 values) are rounded to fp16 again on the way down: one that falls to the other
        # neighbour (2^-11 of its value) is 4e-5 of their norm, and twice that in Adam's second moments.
        tol = {"rel": 4e-4, "max": 4e-3}
    return tol


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=g).mul_(scale)

    def uniform(*shape, lo=-1.0, hi=1.0):
        return torch.rand(*shape, device="cuda", generator=g).mul_(hi - lo).add_(lo)

    def empty(*shape):
        return torch.empty(shape, dtype=torch.float32, device="cuda")

    kind = case["kind"]
    s = {"kind": kind}
    if kind == "gemm":
        M, K, N = case["M"], case["K"], case["N"]
        A, B, s["C"] = uniform(M, K), uniform(*((N, K) if case["b_trans"] else (K, N))), empty(M, N)
        s["call"] = capi.prepare_gemm(A, B, s["C"], b_trans=case["b_trans"])
    elif kind == "linear":
        S, I, O = case["samples"], case["inputs"], case["outputs"]
        x, W, b, s["y"] = normal(S, I), uniform(O, I), uniform(O, lo=-0.03, hi=0.03), empty(S, O)
        W.mul_(math.sqrt(6.0 / I))
        s["call"] = capi.prepare_gemm(x, W, s["y"], b_trans=True, bias=b, bias_strides=(0, 1), relu=True,
                                      prepared_b=capi.Prepared() if case["kept"] else None)
    elif kind == "linear_train":
        S, I, O = case["samples"], case["inputs"], case["outputs"]
        s.update(x=normal(S, I), W=uniform(O, I).mul_(math.sqrt(6.0 / I)), b=uniform(1, 1, O, 1, lo=-0.03, hi=0.03),
                 dy=normal(S, 1, O, 1), y=empty(S, O), dx=empty(S, 1, I, 1), dW=empty(1, 1, O, I), db=empty(1, 1, O, 1))
    elif kind == "batched":
        n, c, M, K, N = (case[k] for k in ("n", "c", "M", "K", "N"))
        s.update(A=normal(n, c, M, K, scale=K ** -0.5), B=normal(n, c, K, N, scale=K ** -0.5), C=empty(n, c, M, N))
    elif kind in ("conv", "conv_train"):
        n, C, H, W, O, K = (case[k] for k in ("n", "C", "H", "W", "O", "K"))
        Ho, Wo = _outputs(case)
        s.update(K=K, stride=case["stride"], pad=case["pad"], x=normal(n, C, H, W),
                 w=normal(n if case["per_sample"] else 1, 1, C * K * K, O, scale=math.sqrt(2.0 / (C * K * K))), y=empty(n, O, Ho, Wo))
        if case["per_sample"] or kind == "conv_train":
            s.update(b=uniform(1, 1, Ho * Wo, O, lo=-0.03, hi=0.03), bias_strides=(O, 1))
        else:
            s.update(b=uniform(O, lo=-0.03, hi=0.03), bias_strides=(0, 1))
        if kind == "conv":
            s["handle"] = capi.Prepared() if case["kept"] else None
        else:
            s.update(dy=normal(n, O, Ho, Wo), dx=empty(n, C, H, W), dw=torch.empty_like(s["w"]), db=torch.empty_like(s["b"]))
    else:
        n, H, W = case["n"], case["H"], case["W"]
        hp, wp = _readme_sizes(case)
        params = [uniform(n, 1, 27, 1, lo=0.0, hi=2.0 / 27), uniform(1, 1, H * W, 1, lo=0.0, hi=2.0 / (H * W) + 1e-4),
                  uniform(n, 1, 9, 1, lo=0.0, hi=2.0 / 9), uniform(1, 1, H * W, 1, lo=0.0, hi=2.0 / (H * W) + 1e-4),
                  uniform(1, 1, 16, hp * wp, lo=0.0, hi=2.0 / (16 * hp * wp) + 1e-4), uniform(1, 1, 16, 1, lo=0.0, hi=0.125)]
        labels = torch.full((1, 1, 16, 1), 0.02, device="cuda")
        labels[0, 0, seed % 16, 0] = 0.7
        s.update(params=params, grads=[torch.empty_like(p) for p in params], m=[torch.zeros_like(p) for p in params],
                 v=[torch.zeros_like(p) for p in params], step=0, lr=0.25 / (hp * wp), x=uniform(n, 3, H, W, lo=0.0, hi=1.0),
                 labels=labels, y1=empty(n, 1, H, W), y2=empty(n, 1, H, W), y4=empty(n, 16), dpool=empty(n, 1, hp * wp, 1),
                 d2=empty(n, 1, H, W), d1=empty(n, 1, H, W))
    return s


def run(s):
    return _RUN[s["kind"]](s)


def _gemm(s):
    s["call"]()
    return s["C"]


def _linear(s):
    s["call"]()
    return s["y"]


def _linear_train(s):
    x, W, b, y = s["x"], s["W"], s["b"], s["y"]
    (S, I), O = x.shape, W.shape[0]
    capi.gemm(x, W, b_trans=True, bias=b, bias_strides=(0, 1), relu=True, out=y)
    dz = capi.relu_backward(y.view(S, 1, O, 1), s["dy"])
    capi.fill_many([s["dW"], s["dx"], s["db"]], 0.0)
    capi.add_backward(s["db"], dz)
    capi.matmul_backward(s["dW"], s["dx"], W.view(1, 1, O, I), x.view(S, 1, I, 1), dz)
    capi.sgd_step_many([W, b], [s["dW"], s["db"]], 1e-7)
    return y, s["dx"], s["dW"], s["db"], W, b


def _batched(s):
    return capi.tensorcore_gemm(s["A"], s["B"], out=s["C"])


def _conv(s):
    return capi.conv2d_forward(s["x"], s["w"], s["b"], s["K"], s["K"], s["stride"], s["pad"], bias_strides=s["bias_strides"],
                               relu=True, out=s["y"], prepared_w=s["handle"])


def _conv_train(s):
    x, w, K, stride, pad = s["x"], s["w"], s["K"], s["stride"], s["pad"]
    y = capi.conv2d_forward(x, w, s["b"], K, K, stride, pad, bias_strides=s["bias_strides"], relu=True, out=s["y"])
    capi.fill_many([s["dw"], s["db"]], 0.0)
    dz = capi.conv2d_backward_relu_bias(s["db"], y, s["dy"])
    capi.conv2d_backward_weights(s["dw"], x, dz, K, K, stride, pad)
    capi.conv2d_backward_data(s["dx"], dz, w, K, K, stride, pad, accumulate=False)
    return y, s["dw"], s["db"], s["dx"]


def _readme_step(s):
    w1, b1, w2, b2, W, b = s["params"]
    dw1, db1, dw2, db2, dW, db = s["grads"]
    n = s["x"].shape[0]
    fan_in = W.shape[3]
    # forward
    y1 = capi.conv2d_forward(s["x"], w1, b1, 3, 3, 1, 1, bias_strides=(1, 1), relu=True, out=s["y1"])
    y2 = capi.conv2d_forward(y1, w2, b2, 3, 3, 1, 1, bias_strides=(1, 1), out=s["y2"])
    pooled = capi.avgpool2d(y2, 5, 2, 0)
    y4 = capi.gemm(pooled.view(n, fan_in), W.view(16, fan_in), b_trans=True, bias=b, bias_strides=(0, 1), out=s["y4"])
    p = capi.softmax(y4.view(n, 1, 16, 1))
    target = capi.expand(s["labels"], n)
    loss = capi.bce_loss(p, target)
    # backward
    capi.fill_many(s["grads"] + [s["dpool"]], 0.0)
    dz = capi.softmax_backward(p, capi.bce_backward(p, target))
    capi.add_backward(db, dz)
    capi.matmul_backward(dW, s["dpool"], W, pooled.view(n, 1, fan_in, 1), dz)
    capi.avgpool2d_backward(s["d2"], s["dpool"].view(pooled.shape), 5, 2, 0, overwrite=True)
    capi.conv2d_backward_bias(db2, s["d2"])
    capi.conv2d_backward_weights(dw2, y1, s["d2"], 3, 3, 1, 1)
    capi.conv2d_backward_data(s["d1"], s["d2"], w2, 3, 3, 1, 1, accumulate=False)
    d1 = capi.conv2d_backward_relu_bias(db1, y1, s["d1"])
    capi.conv2d_backward_weights(dw1, s["x"], d1, 3, 3, 1, 1)
    # Adam counts its calls: the tensors of one update have consecutive step counts
    first = s["step"]
    s["step"] += len(s["params"])
    capi.adam_step_many(s["params"], s["m"], s["v"], s["grads"], [first + k + 1 for k in range(len(s["params"]))], s["lr"], 0.9, 0.999, 1e-8)
    return {"loss": loss, "p": p, "grads": s["grads"], "params": s["params"], "m": s["m"], "v": s["v"]}


_RUN = {"gemm": _gemm, "linear": _linear, "linear_train": _linear_train, "batched": _batched, "conv": _conv, "conv_train": _conv_train,
        "readme_step": _readme_step}

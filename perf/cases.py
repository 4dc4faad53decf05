"""The work that a program built on this framework spends its time in, as cases that can be timed.

Four families, each through `neurotensor_amd.functional`:

  matmult         C = op(a).op(b), single and batched, every storage form, floating and integer types
  linear          y = x.W + bias (with or without the clamp of relu): inference on few or many rows
  linear_train    a Linear layer's step: forward, gradient of the input, gradient of the weight
  conv_train      a convolution layer's step over one to three axes, plain or transposed: forward and both gradients

`listed()` names twelve of them, `draw(rng)` gives more of the same ranges.
"""
import math

import torch

from neurotensor_amd import functional as F

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32, "float64": torch.float64,
          "int8": torch.int8, "int16": torch.int16, "int32": torch.int32, "int64": torch.int64}
INTEGERS = ("int8", "int16", "int32", "int64")
# Orders of magnitude of what one card does with each type (operations a second): they only bound how much work is drawn.
RATE = {"float16": 1.0e15, "bfloat16": 1.0e15, "float32": 1.2e14, "float64": 6.0e13, "int8": 1.5e15, "int16": 3.0e14, "int32": 9.0e13, "int64": 2.5e13}


def listed():
    return [
        # The step of a small classifier's hidden layer (28 x 28 inputs, one minibatch): three short calls, the launches count.
        {"name": "linear_train_small_fp32", "op": "linear_train", "dtype": "float32", "rows": 64, "k": 784, "n": 128, "weight_t": False},
        # The step of a wide feed-forward layer: the largest product that bench.py's configurations hold.
        {"name": "linear_train_bf16", "op": "linear_train", "dtype": "bfloat16", "rows": 8192, "k": 4096, "n": 11008, "weight_t": True},
        # The same layer at inference on sixteen rows (decode): the weight is read once, memory is the bound.
        {"name": "linear_decode_bf16", "op": "linear", "dtype": "bfloat16", "rows": 16, "k": 4096, "n": 11008, "weight_t": True, "relu": False},
        # The headline product.
        {"name": "matmult_bf16_4096", "op": "matmult", "dtype": "bfloat16", "batch": 1, "m": 4096, "k": 4096, "n": 4096,
         "ta": False, "tb": False, "shared_b": False},
        # A batched product with a transposed right operand (attention scores, per-sample products).
        {"name": "matmult_fp32_batch", "op": "matmult", "dtype": "float32", "batch": 32, "m": 1024, "k": 768, "n": 1024,
         "ta": False, "tb": True, "shared_b": False},
        # Sizes off every tile and every 16-byte boundary, as data and not a layer's author gives them.
        {"name": "matmult_fp16_odd", "op": "matmult", "dtype": "float16", "batch": 1, "m": 1023, "k": 1537, "n": 2049,
         "ta": False, "tb": False, "shared_b": False},
        # The integer batch of bench.py's configurations: exact, wrapping sums.
        {"name": "matmult_int32_batch", "op": "matmult", "dtype": "int32", "batch": 8, "m": 1024, "k": 1024, "n": 1024,
         "ta": False, "tb": False, "shared_b": False},
        # Double precision at the size that the reference's own speed test takes.
        {"name": "matmult_fp64_1000", "op": "matmult", "dtype": "float64", "batch": 1, "m": 1000, "k": 1000, "n": 1000,
         "ta": False, "tb": False, "shared_b": False},
        # A residual network's 3 x 3 layer in 16 bits.
        {"name": "conv2d_train_bf16", "op": "conv_train", "dtype": "bfloat16", "axes": 2, "batch": 64, "cin": 256, "cout": 256,
         "size": 56, "kernel": 3, "stride": 1, "groups": 1, "transposed": False},
        # An image network's first layer: three channels, a wide kernel, stride 2.
        {"name": "conv2d_train_rgb_fp32", "op": "conv_train", "dtype": "float32", "axes": 2, "batch": 32, "cin": 3, "cout": 64,
         "size": 224, "kernel": 7, "stride": 2, "groups": 1, "transposed": False},
        # A volumetric network's layer.
        {"name": "conv3d_train_fp32", "op": "conv_train", "dtype": "float32", "axes": 3, "batch": 4, "cin": 32, "cout": 64,
         "size": 32, "kernel": 3, "stride": 1, "groups": 1, "transposed": False},
        # A decoder's layer that doubles the image.
        {"name": "conv_transpose2d_train_fp16", "op": "conv_train", "dtype": "float16", "axes": 2, "batch": 32, "cin": 128, "cout": 64,
         "size": 28, "kernel": 4, "stride": 2, "groups": 1, "transposed": True},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm; half of them whole multiples of 64, a quarter of 8, a quarter as they fall."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice((64, 64, 8, 1))
    return min(hi, max(lo, (v + step // 2) // step * step if v >= step else v))


def _drawn(rng):
    op = rng.choice(("matmult", "matmult", "linear", "linear_train", "conv_train", "conv_train"))
    if op == "matmult":
        dtype = rng.choice(("float32", "float32", "bfloat16", "bfloat16", "float16", "float64", "int32", "int8", "int16", "int64"))
        batch = rng.choice((1, 1, _size(rng, 2, 64)))
        return {"op": op, "dtype": dtype, "batch": batch, "m": _size(rng, 32, 4096), "k": _size(rng, 32, 4096), "n": _size(rng, 32, 4096),
                "ta": rng.random() < 0.25, "tb": rng.random() < 0.4, "shared_b": batch > 1 and rng.random() < 0.25}
    dtype = rng.choice(("float32", "bfloat16", "float16"))
    if op == "linear":
        return {"op": op, "dtype": dtype, "rows": rng.choice((_size(rng, 1, 64), _size(rng, 64, 4096))), "k": _size(rng, 64, 8192),
                "n": _size(rng, 64, 11008), "weight_t": rng.random() < 0.5, "relu": rng.random() < 0.5}
    if op == "linear_train":
        return {"op": op, "dtype": dtype, "rows": _size(rng, 32, 8192), "k": _size(rng, 64, 4096), "n": _size(rng, 64, 11008),
                "weight_t": rng.random() < 0.5}
    axes = rng.choice((1, 2, 2, 2, 3))
    transposed = rng.random() < 0.25
    stride = 2 if transposed else rng.choice((1, 1, 2))
    kernel = rng.choice((2, 4)) if transposed else rng.choice((1, 3, 3, 5, 7) if axes < 3 else (1, 3, 3))
    groups = rng.choice((1, 1, 1, 2, 4))
    if groups == 1 and not transposed and rng.random() < 0.2:
        cin = rng.choice((1, 3))
    else:
        cin = rng.choice((16, 24, 32, 48, 64, 96, 128, 192, 256))
    return {"op": op, "dtype": dtype, "axes": axes, "batch": _size(rng, 1, 64), "cin": cin,
            "cout": rng.choice((16, 32, 48, 64, 96, 128, 192, 256)),
            "size": _size(rng, 128, 8192) if axes == 1 else _size(rng, 7, 224) if axes == 2 else _size(rng, 8, 48),
            "kernel": kernel, "stride": stride, "groups": groups, "transposed": transposed}


def draw(rng):
    """One more case: half of what the largest listed case costs at the rates above, at most."""
    most = max(_cost(c) for c in listed())
    while True:
        c = _drawn(rng)
        if c["op"] == "conv_train" and c["size"] < c["kernel"]:
            continue
        if _cost(c) <= 0.5 * most and work(c)["bytes"] <= 2e9:
            return c


def _cost(c):
    w = work(c)
    return w["flops"] / RATE[c["dtype"]] + w["bytes"] / 4e12


def _conv_geometry(c):
    """(padding, output size along each axis)."""
    k, s = c["kernel"], c["stride"]
    if c["transposed"]:
        p = (k - s) // 2
        return p, (c["size"] - 1) * s - 2 * p + k
    p = k // 2
    return p, (c["size"] + 2 * p - k) // s + 1


def _values(shape, dtype, gen, scale=1.0):
    if dtype in INTEGERS:
        lo, hi = (-128, 128) if dtype == "int8" else (-8, 9)
        return torch.randint(lo, hi, shape, device="cuda", dtype=DTYPES[dtype], generator=gen)
    if dtype == "float64":
        return torch.randn(shape, device="cuda", dtype=torch.float64, generator=gen) * scale
    return (torch.randn(shape, device="cuda", generator=gen) * scale).to(DTYPES[dtype])


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    c, dt = dict(case), case["dtype"]
    if c["op"] == "matmult":
        lead = (c["batch"],) if c["batch"] > 1 else ()
        a = _values(lead + ((c["k"], c["m"]) if c["ta"] else (c["m"], c["k"])), dt, gen)
        b = _values((() if c["shared_b"] else lead) + ((c["n"], c["k"]) if c["tb"] else (c["k"], c["n"])), dt, gen)
        return {"case": c, "a": a, "b": b}
    if c["op"] in ("linear", "linear_train"):
        k, n = c["k"], c["n"]
        state = {"case": c, "x": _values((c["rows"], k), dt, gen), "w": _values((n, k) if c["weight_t"] else (k, n), dt, gen, k ** -0.5),
                 "bias": _values((n,), dt, gen, 0.1)}
        if c["op"] == "linear_train":
            state["dy"] = _values((c["rows"], n), dt, gen)
        return state
    p, out = _conv_geometry(c)
    k, axes, g = c["kernel"], c["axes"], c["groups"]
    shape = (c["cin"], c["cout"] // g) if c["transposed"] else (c["cout"], c["cin"] // g)
    fan = c["cin"] // g * k ** axes
    return {"case": c, "x": _values((c["batch"], c["cin"]) + (c["size"],) * axes, dt, gen), "w": _values(shape + (k,) * axes, dt, gen, fan ** -0.5),
            "dy": _values((c["batch"], c["cout"]) + (out,) * axes, dt, gen), "padding": p}


_FORWARD = {(1, False): F.conv1d, (2, False): F.conv2d, (3, False): F.conv3d,
            (1, True): F.conv_transpose1d, (2, True): F.conv_transpose2d, (3, True): F.conv_transpose3d}
_BACKWARD = {(1, False): F.conv1d_backward, (2, False): F.conv2d_backward, (3, False): F.conv3d_backward,
             (1, True): F.conv_transpose1d_backward, (2, True): F.conv_transpose2d_backward, (3, True): F.conv_transposend_backward}


def run(state):
    c = state["case"]
    if c["op"] == "matmult":
        return F.matmult(state["a"], state["b"], None, c["ta"], c["tb"])
    if c["op"] == "linear":
        layer = F.linear_relu if c["relu"] else F.linear
        return layer(state["x"], state["w"], state["bias"], False, c["weight_t"])
    if c["op"] == "linear_train":
        x, w, dy = state["x"], state["w"], state["dy"]
        y = F.linear(x, w, state["bias"], False, c["weight_t"])
        if c["weight_t"]:                       # W stored [out, in]: dX = dY.W, dW = dY^T.X
            return {"y": y, "dx": F.matmult(dy, w), "dw": F.matmult(dy, x, None, True, False)}
        return {"y": y, "dx": F.matmult(dy, w, None, False, True), "dw": F.matmult(x, dy, None, True, False)}
    kind = (c["axes"], c["transposed"])
    options = {"stride": c["stride"], "padding": state["padding"], "groups": c["groups"]}
    y = _FORWARD[kind](state["x"], state["w"], **options)
    dx, dw = _BACKWARD[kind](state["x"], state["w"], state["dy"], **options)
    return {"y": y, "dx": dx, "dw": dw}


def work(case):
    """Bytes with each input read once and each output written once; operations of the sums that define the outputs."""
    c, es = case, DTYPES[case["dtype"]].itemsize
    if c["op"] == "matmult":
        m, k, n, b = c["m"], c["k"], c["n"], c["batch"]
        return {"bytes": es * (b * m * k + (1 if c["shared_b"] else b) * k * n + b * m * n), "flops": 2 * b * m * k * n}
    if c["op"] in ("linear", "linear_train"):
        m, k, n = c["rows"], c["k"], c["n"]
        once = m * k + k * n + m * n
        return {"bytes": es * (n + (once if c["op"] == "linear" else 2 * once)), "flops": (2 if c["op"] == "linear" else 6) * m * k * n}
    _, out = _conv_geometry(c)
    x, y = c["batch"] * c["cin"] * c["size"] ** c["axes"], c["batch"] * c["cout"] * out ** c["axes"]
    w = c["cin"] * c["cout"] // c["groups"] * c["kernel"] ** c["axes"]
    positions = c["batch"] * (c["size"] if c["transposed"] else out) ** c["axes"]      # each sees every weight once
    return {"bytes": es * 2 * (x + y + w), "flops": 6 * positions * w}


# The largest relative error between two correct implementations at one precision: about four times what the results show against the
# same path in 64 bits (Float64: against the sum in another order).  Seen: BFloat16 1.7e-3 (2.4e-3 for a weight gradient summed over
# images), Float16 2.1e-4 (2.9e-4), Float32 1e-7 to 3.2e-6, Float64 3.9e-16 at k = 1000.
_REL = {"bfloat16": 8e-3, "float16": 1e-3, "float32": 1e-5, "float64": 4e-15}


def tolerance(case):
    if case["dtype"] in INTEGERS:
        return "exact"
    return {"rel": _REL[case["dtype"]]}

"""The convolutions that a user of this lab runs, as measurable cases.

A case is one convolution layer (``kind`` "conv") through ``launch`` (int32
output) or ``launch_requant`` (int8 output), on tensors and a stream that the
program owns, or one residual-style bottleneck (``kind`` "block"): channel-major
activations in, three layers, channel-major accumulators out.  The layers are
those of ``workloads/baseline.csv`` and ``workloads/reference.csv``, at the
batch sizes of those tables or a generic one.

``prepare`` holds what such a program keeps: the tensors, the chosen kernel,
the output and the workspace; ``run`` is one pass.  All results are whole
numbers, so the tolerance is "exact" everywhere.
"""
from __future__ import annotations

import math

import torch

import int8_kernel_lab_amd as lab

CONV_FIELDS = ("n", "h", "w", "c", "k", "r", "s", "pad_h", "pad_w",
               "stride_h", "stride_w", "dilation_h", "dilation_w")

# The largest listed layer: no drawn case does more operations or moves more bytes.
MOST_OPS = 2 * (16 * 256 * 256) * 256 * (9 * 256)
MOST_BYTES = 16 * 256 * 256 * (256 + 4 * 256)


def _conv(name, out, n, h, w, c, k, r, s, pad_h=0, pad_w=0, stride_h=1, stride_w=1,
          dilation_h=1, dilation_w=1):
    case = dict(zip(CONV_FIELDS, (n, h, w, c, k, r, s, pad_h, pad_w, stride_h, stride_w,
                                  dilation_h, dilation_w)))
    return {"name": name, "kind": "conv", "out": out, **case}


def listed():
    return [
        # One image through a late 3x3 layer: the smallest call, where the
        # launch and the host's share of it count.
        _conv("b1_14x14x256_3x3", "int32", 1, 14, 14, 256, 256, 3, 3, 1, 1),
        # The 3x3 layer of a batch of 32 in the middle of a ResNet.
        _conv("b32_28x28x128_3x3", "int32", 32, 28, 28, 128, 128, 3, 3, 1, 1),
        # A downsampling layer of a quantized network: stride 2, int8 output.
        _conv("b32_56x56x128_3x3_s2_int8", "int8", 32, 56, 56, 128, 256, 3, 3, 1, 1, 2, 2),
        # The 1x1 reduction of a bottleneck at batch 64: bandwidth.
        _conv("b64_56x56x256_1x1", "int32", 64, 56, 56, 256, 64, 1, 1),
        # Few pixels and a long reduction: the last stage of a network.
        _conv("b8_7x7x2048_3x3", "int32", 8, 7, 7, 2048, 512, 3, 3, 1, 1),
        # A dilated layer, as in segmentation networks.
        _conv("b8_64x64x256_3x3_d2", "int32", 8, 64, 64, 256, 256, 3, 3, 2, 2, 1, 1, 2, 2),
        # The two halves of a separated filter are shaped like this one.
        _conv("b8_128x128x64_1x3", "int32", 8, 128, 128, 64, 128, 1, 3, 0, 1),
        # A detection head: an output channel count that is no multiple of 4.
        _conv("b1_256x256x64_k255", "int32", 1, 256, 256, 64, 255, 3, 3, 1, 1),
        # The 7x7 stride-2 stem of a quantized network, channels padded to 32.
        _conv("b16_224x224x32_7x7_s2_int8", "int8", 16, 224, 224, 32, 64, 7, 7, 3, 3, 2, 2),
        # The largest layers of the table: throughput, with int32 and int8 output.
        _conv("b16_256x256x256_3x3", "int32", 16, 256, 256, 256, 256, 3, 3, 1, 1),
        _conv("b16_256x256x256_5x5_s2_int8", "int8", 16, 256, 256, 256, 256, 5, 5, 2, 2, 2, 2),
        # A bottleneck of a quantized network, between channel-major tensors.
        {"name": "b32_56x56x256_bottleneck", "kind": "block", "n": 32, "h": 56, "w": 56,
         "c": 256, "mid": 64},
    ]


# ---- drawn cases -------------------------------------------------------------

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(("3x3", "3x3", "3x3", "down", "1x1", "1x1", "dilated", "long", "stem",
                       "deep", "block"))
    n = _log(rng, 1, 32)
    c = 16 * _log(rng, 2, 32)
    k = _log(rng, 32, 512)
    if rng.random() < 0.7:
        k = 32 * max(1, round(k / 32))
    if rng.random() < 0.6:
        c = 64 * max(1, round(c / 64))
    h = _log(rng, 7, 256)
    w = h if rng.random() < 0.6 else _log(rng, 7, 256)
    if kind == "block":
        return {"kind": "block", "n": n, "h": _log(rng, 7, 64), "w": _log(rng, 7, 64),
                "c": 64 * rng.randint(1, 8), "mid": 64 * rng.randint(1, 4)}
    out = rng.choice(("int32", "int8"))
    if kind == "3x3":
        shape = (n, h, w, c, k, 3, 3, 1, 1)
    elif kind == "down":
        r = rng.choice((3, 3, 5))
        shape = (n, h, w, c, k, r, r, r // 2, r // 2, 2, 2)
    elif kind == "1x1":
        shape = (_log(rng, 1, 64), h, w, c, k, 1, 1)
    elif kind == "dilated":
        d = rng.choice((2, 2, 3))
        shape = (n, h, w, c, k, 3, 3, d, d, 1, 1, d, d)
    elif kind == "long":
        shape = (n, h, w, c, k, 1, 3, 0, 1) if rng.random() < 0.5 else (n, h, w, c, k, 3, 1, 1, 0)
    elif kind == "stem":
        r, st = rng.choice(((7, 2), (4, 4), (3, 1), (3, 2)))
        shape = (n, _log(rng, 64, 416), _log(rng, 64, 416), 32, 32 * rng.randint(1, 4), r, r,
                 (r - 1) // 2 if st < r else 0, (r - 1) // 2 if st < r else 0, st, st)
    else:
        shape = (_log(rng, 1, 8), rng.randint(5, 14), rng.randint(5, 14),
                 128 * rng.randint(4, 16), 64 * rng.randint(2, 16), *rng.choice(
                     ((3, 3, 1, 1), (1, 1, 0, 0))))
    case = _conv("", out, *shape)
    del case["name"]
    return case


def draw(rng):
    while True:
        case = _draw_once(rng)
        total = work(case)
        if 1e7 < total["flops"] <= MOST_OPS and total["bytes"] <= MOST_BYTES:
            return case


# ---- one case ------------------------------------------------------------------

def _layers(case):
    """(shape, output type) of the case's convolutions, in order."""
    if case["kind"] == "conv":
        return [(lab.ConvShape(*[case[f] for f in CONV_FIELDS]), case["out"])]
    n, h, w, c, mid = (case[f] for f in ("n", "h", "w", "c", "mid"))
    return [(lab.ConvShape(n, h, w, c, mid, 1, 1), "int8"),
            (lab.ConvShape(n, h, w, mid, mid, 3, 3, 1, 1), "int8"),
            (lab.ConvShape(n, h, w, mid, c, 1, 1), "int32")]


ZERO_POINT = 3


def _inputs(case, seed):
    """The case's tensors from the seed: int8 over the whole range, biases of
    20 bits, and per-channel scales that spread the result over int8."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def ints(lo, hi, shape, dtype):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=dtype)

    layers = []
    for shape, out in _layers(case):
        layer = {"w": ints(-128, 128, (shape.k, shape.r, shape.s, shape.c), torch.int8),
                 "b": ints(-(1 << 20), (1 << 20) + 1, (shape.k,), torch.int32)}
        if out == "int8":
            # scale = mult / 2^shift: a third of int8's range for a sum's
            # standard deviation, and up to twice that by channel
            deviation = 5461.0 * math.sqrt(shape.r * shape.s * shape.c)
            layer["mult"] = ints(1 << 30, (1 << 31) - 1, (shape.k,), torch.int32)
            low = round(30.5 + math.log2(deviation / 42.0))
            layer["shift"] = ints(low - 1, low + 1, (shape.k,), torch.int32)
        layers.append(layer)
    first = _layers(case)[0][0]
    order = (first.n, first.c, first.h, first.w) if case["kind"] == "block" else \
        (first.n, first.h, first.w, first.c)
    return ints(-128, 128, order, torch.int8), layers


def _plan(shape, out, x, layer):
    """A layer's plan: output, workspace and the pointers of its call."""
    y = torch.empty(shape.output_shape, device="cuda",
                    dtype=torch.int8 if out == "int8" else torch.int32)
    name = lab.dispatch(shape)
    nbytes = lab.requant_workspace_bytes(shape) if out == "int8" else lab.workspace_bytes(name, shape)
    ws = torch.empty(max(nbytes, 1), device="cuda", dtype=torch.uint8)
    return {"shape": shape, "out": out, "name": name, "x": x, "y": y, "ws": ws, "ws_bytes": nbytes,
            **layer}


def prepare(case, seed):
    x, layers = _inputs(case, seed)
    shapes = _layers(case)
    state = {"kind": case["kind"], "x": x, "plans": []}
    if case["kind"] == "block":
        first = shapes[0][0]
        state["nhwc"] = torch.empty((first.n, first.h, first.w, first.c), device="cuda",
                                    dtype=torch.int8)
        x = state["nhwc"]
    for (shape, out), layer in zip(shapes, layers):
        plan = _plan(shape, out, x, layer)
        state["plans"].append(plan)
        x = plan["y"]
    if case["kind"] == "block":
        last = shapes[-1][0]
        state["y"] = torch.empty((last.n, last.k, last.h, last.w), device="cuda",
                                 dtype=torch.int32)
    return state


def _launch(p, stream):
    ws = p["ws"].data_ptr() if p["ws_bytes"] else None
    if p["out"] == "int8":
        lab.launch_requant(p["shape"], p["x"].data_ptr(), p["w"].data_ptr(), p["b"].data_ptr(),
                           p["mult"].data_ptr(), p["shift"].data_ptr(), ZERO_POINT,
                           p["y"].data_ptr(), ws, p["ws_bytes"], stream)
    else:
        lab.launch(p["name"], p["shape"], p["x"].data_ptr(), p["w"].data_ptr(), p["b"].data_ptr(),
                   p["y"].data_ptr(), ws, p["ws_bytes"], stream)


def run(state):
    stream = torch.cuda.current_stream().cuda_stream
    if state["kind"] == "conv":
        _launch(state["plans"][0], stream)
        return state["plans"][0]["y"]
    first, last = state["plans"][0]["shape"], state["plans"][-1]["shape"]
    lab.nchw_to_nhwc(state["x"].data_ptr(), state["nhwc"].data_ptr(), first.n, first.c, first.h,
                     first.w, stream)
    for p in state["plans"]:
        _launch(p, stream)
    lab.nhwk_to_nkhw(state["plans"][-1]["y"].data_ptr(), state["y"].data_ptr(), last.n, last.h,
                     last.w, last.k, stream)
    return state["y"]


def work(case):
    """Operations 2*M*N*K with padded taps; input, filters and per-channel
    parameters read once, the result written once."""
    ops, nbytes = 0, 0
    layers = _layers(case)
    for i, (shape, out) in enumerate(layers):
        g = shape.geometry()
        ops += shape.ops()
        nbytes += g.filter_elements + (12 if out == "int8" else 4) * shape.k
        if i == 0:
            nbytes += g.input_elements
        if i == len(layers) - 1:
            nbytes += g.output_elements * (1 if out == "int8" else 4)
    return {"bytes": nbytes, "flops": ops}


def tolerance(case):
    return "exact"


# ---- the same in 64 bits -------------------------------------------------------

def _exact_conv(shape, x, layer):
    """int64 NHWK sums: every product and sum below 2^53, so float64 is exact."""
    oh, ow = shape.out_h, shape.out_w
    xp = torch.nn.functional.pad(x, (0, 0, shape.pad_w, shape.pad_w, shape.pad_h, shape.pad_h))
    y = layer["b"].double().expand(shape.n * oh * ow, shape.k).contiguous()
    for fy in range(shape.r):
        for fx in range(shape.s):
            y0, x0 = fy * shape.dilation_h, fx * shape.dilation_w
            rows = xp[:, y0:y0 + (oh - 1) * shape.stride_h + 1:shape.stride_h,
                      x0:x0 + (ow - 1) * shape.stride_w + 1:shape.stride_w]
            y.addmm_(rows.reshape(-1, shape.c).double(),
                     layer["w"][:, fy, fx].double().t().contiguous())
    return y.round_().to(torch.int64).reshape(shape.n, oh, ow, shape.k)


def _exact_requant(acc, layer):
    """clamp(zp + round(acc * mult / 2^shift)), ties away from zero, in int64."""
    p = acc * layer["mult"].long()
    s = layer["shift"].long()
    half = torch.ones_like(s) << (s - 1)
    q = ((p.abs() + half) >> s) * p.sign()
    return (q + ZERO_POINT).clamp(-128, 127).to(torch.int8)


def exact(case, seed):
    x, layers = _inputs(case, seed)
    if case["kind"] == "block":
        x = x.permute(0, 2, 3, 1).contiguous()
    for (shape, out), layer in zip(_layers(case), layers):
        acc = _exact_conv(shape, x, layer)
        x = _exact_requant(acc, layer) if out == "int8" else acc.to(torch.int32)
    return x.permute(0, 3, 1, 2).contiguous() if case["kind"] == "block" else x

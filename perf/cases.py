"""The workloads by which the speed of `ruy_amd.api.mul` is judged.

`listed()` names twelve calls, from the smallest a quantized network makes to
the largest the benchmark times; `draw()` gives more of the same ranges. A case
is one product: operand types, sizes, storage orders, padding of the strides,
zero points and the options of MulParams.

Except for the host-memory cases the program has its matrices in device
memory, launches on torch's current stream and lets calls return once they are
enqueued, as bench.py does.
"""
import math

import torch

from ruy_amd import _structs as S
from ruy_amd import api
from ruy_amd import workloads as W

_TYPES = {
    "uint8": (S.U8, torch.uint8), "int8": (S.I8, torch.int8), "int16": (S.I16, torch.int16),
    "int32": (S.I32, torch.int32), "f32": (S.F32, torch.float32),
}
_ORDERS = {"col": api.Order.kColMajor, "row": api.Order.kRowMajor}

# Operands as a fully connected or 1x1 convolution layer has them: weights by
# rows, activations by columns (both depth-contiguous), destination by columns.
_LAYER = {"lhs_order": "row", "rhs_order": "col", "dst_order": "col", "pad": 0,
          "lhs_zero": 0, "rhs_zero": 0, "dst_zero": 0, "bias": True, "perchannel": False,
          "relu6": False, "cached_lhs": False, "host": False}


def _case(name, types, m, k, n, **options):
    lhs, rhs, dst = types.split("*")
    case = dict(_LAYER, lhs=lhs, rhs=rhs, dst=dst, m=m, k=k, n=n, **options)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest layer: one call is a launch and little else.
        _case("int8 256", "int8*int8*int8", 256, 256, 256, rhs_zero=-3, dst_zero=5),
        # A 1x1 convolution over a 14x14 image, per-channel quantization.
        _case("int8 1x1 conv", "int8*int8*int8", 1024, 1024, 196, rhs_zero=-128, dst_zero=-128, perchannel=True),
        # The first layer of an image network: 7x7x3 windows (an odd depth)
        # over 112x112 positions, asymmetric uint8 throughout.
        _case("uint8 7x7 conv", "uint8*uint8*uint8", 64, 147, 12544, lhs_zero=117, rhs_zero=128, dst_zero=121),
        # An ordinary layer at a large batch.
        _case("int8 2048", "int8*int8*int8", 2048, 2048, 2048, rhs_zero=-3, dst_zero=5),
        # A general product: both operands as BLAS callers hold them (by
        # columns, one of them transposed for the kernels), strides that are
        # no multiple of anything, row-major destination, both zero points.
        _case("int8 by columns", "int8*int8*int8", 1000, 1500, 700, lhs_order="col", dst_order="row", pad=1,
              lhs_zero=4, rhs_zero=-3, dst_zero=5),
        # The benchmark's headline.
        _case("int8 8192", "int8*int8*int8", 8192, 8192, 8192, rhs_zero=-3, dst_zero=5),
        # fp32 layers: a square one with its activation, and a ragged one.
        _case("f32 1024", "f32*f32*f32", 1024, 1024, 1024, relu6=True),
        _case("f32 ragged", "f32*f32*f32", 1537, 1111, 2051),
        # 16-bit activations against 8-bit weights.
        _case("int8 int16", "int8*int16*int16", 2048, 2048, 512),
        # One token through a large layer whose weights the cache holds.
        _case("int8 gemv 16384", "int8*int8*int32", 16384, 16384, 1, rhs_zero=7, bias=False, cached_lhs=True),
        # A few tokens through an fp32 layer.
        _case("f32 skinny", "f32*f32*f32", 4096, 4096, 4),
        # The caller of a CPU library: everything in host memory, the weights
        # constant and cached, activations and results new on each call.
        _case("int8 1x1 conv from host", "int8*int8*int8", 1024, 1024, 196, rhs_zero=-128, dst_zero=-128,
              perchannel=True, cached_lhs=True, host=True),
    ]


# fp32 runs at a sixteenth of the rate of int8, int8 x int16 at half of it.
_MOST_FLOPS = {"int8": 1.0e12, "uint8": 1.0e12, "f32": 4.0e10, "int8*int16": 2.0e11}


def _spread(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]; every other one is a
    multiple of 16 as layers mostly have them, the rest are as they fall."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v = (v + 15) // 16 * 16
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["int8", "int8", "int8", "uint8", "uint8", "f32", "f32", "int8*int16", "skinny", "skinny", "host"])
    o = {}
    if kind == "skinny":
        types = rng.choice(["int8*int8*int32", "int8*int8*int8", "f32*f32*f32"])
        m, k, n = _spread(rng, 512, 16384), _spread(rng, 512, 16384), rng.randint(1, 16)
    elif kind == "host":
        types = rng.choice(["int8*int8*int8", "uint8*uint8*uint8", "f32*f32*f32"])
        hi = 512 if types.startswith("f32") else 1024
        m, k, n = _spread(rng, 64, hi), _spread(rng, 64, hi), _spread(rng, 1, hi)
        o["host"] = True
    else:
        types, hi = {"int8": ("int8*int8*int8", 8192), "uint8": ("uint8*uint8*uint8", 4096),
                     "f32": ("f32*f32*f32", 3072), "int8*int16": ("int8*int16*int16", 4096)}[kind]
        m, k, n = _spread(rng, 64, hi), _spread(rng, 64, hi), _spread(rng, 64, 2 * hi)
        while 2.0 * m * k * n > _MOST_FLOPS[kind]:
            n = (n + 1) // 2
    eight_bit = types.startswith(("int8*int8", "uint8"))
    if eight_bit:
        centre = 128 if types.startswith("uint8") else 0
        o["rhs_zero"] = centre + rng.choice([0, -3, 7])
        o["lhs_zero"] = centre + (rng.choice([-11, 0, 4]) if centre else 0)
        if not types.endswith("int32"):
            o["dst_zero"] = centre + rng.choice([-7, 0, 5])
    if types.endswith("int32"):
        o["bias"] = rng.random() < 0.5
    elif types.startswith("f32"):
        o["relu6"] = rng.random() < 0.5
    else:
        o["perchannel"] = rng.random() < 0.5
    o["cached_lhs"] = rng.random() < (0.7 if kind in ("skinny", "host") else 0.1)
    if kind not in ("skinny", "host") and rng.random() < 0.3:
        o["lhs_order"], o["rhs_order"], o["dst_order"] = rng.choice(
            [("col", "col", "col"), ("row", "row", "row"), ("row", "row", "col"), ("col", "col", "row")])
        o["pad"] = rng.randint(0, 1)
    return _case("", types, m, k, n, **o)


def _values(generator, kind, count, weights):
    """Weights over the symmetric range, activations over all of it."""
    where = generator.device
    if kind == "f32":
        return torch.rand(count, generator=generator, device=where).mul_(2).sub_(1)
    lo, hi = S.INT_RANGES[_TYPES[kind][0]]
    if weights and kind == "int8":
        lo += 1
    return torch.randint(lo, hi + 1, (count,), generator=generator, device=where, dtype=_TYPES[kind][1])


def _matrix(kind, rows, cols, order, pad, zero, buffer_of, cached=False):
    layout = api.make_simple_layout(rows, cols, _ORDERS[order])
    layout.stride += pad
    data = buffer_of(api.storage_elements(layout))
    policy = api.CachePolicy.kAlwaysCache if cached else api.CachePolicy.kNeverCache
    return api.Matrix(_TYPES[kind][0], data, layout, zero, policy)


def prepare(case, seed):
    c = case
    where = "cpu" if c["host"] else "cuda"
    g = torch.Generator(device=where)
    g.manual_seed(seed)

    def given(t):
        return t.numpy() if c["host"] else t

    lhs = _matrix(c["lhs"], c["m"], c["k"], c["lhs_order"], c["pad"], c["lhs_zero"],
                  lambda n: given(_values(g, c["lhs"], n, True)), c["cached_lhs"])
    rhs = _matrix(c["rhs"], c["k"], c["n"], c["rhs_order"], c["pad"], c["rhs_zero"],
                  lambda n: given(_values(g, c["rhs"], n, False)))
    dst = _matrix(c["dst"], c["m"], c["n"], c["dst_order"], c["pad"], c["dst_zero"],
                  lambda n: given(torch.zeros(n, dtype=_TYPES[c["dst"]][1], device=where)))

    floats = c["dst"] == "f32"
    params = api.MulParams(S.F32 if floats else S.I32, _TYPES[c["dst"]][0])
    if c["bias"]:
        params.set_bias(given(_values(g, "f32", c["m"], False) if floats else
                              torch.randint(-1000, 1001, (c["m"],), generator=g, device=where, dtype=torch.int32)))
    if c["relu6"]:
        params.set_clamp_min(0.0)
        params.set_clamp_max(6.0)
    if c["dst"] in ("int8", "uint8", "int16"):
        # Scaled so that the results spread over the destination's range.
        spread = {"int8": 74.0, "uint8": 74.0, "int16": 18918.0}
        scale = spread[c["dst"]] / 2 / (spread[c["lhs"]] * spread[c["rhs"]] * math.sqrt(c["k"]))
        fixed, exponent = W.quantize_multiplier(scale)
        if c["perchannel"]:
            params.set_multiplier_fixedpoint_perchannel(given(torch.randint(
                1 << 30, (1 << 31) - 1, (c["m"],), generator=g, device=where, dtype=torch.int32)))
            params.set_multiplier_exponent_perchannel(given(torch.randint(
                exponent - 1, exponent + 2, (c["m"],), generator=g, device=where, dtype=torch.int32)))
        else:
            params.set_multiplier_fixedpoint(fixed)
            params.set_multiplier_exponent(exponent)

    context = api.Context()
    if c["cached_lhs"]:
        context.set_cache_max_bytes(2 << 30)
    if not c["host"]:
        context.set_stream(torch.cuda.current_stream().cuda_stream)
        context.set_synchronous(False)
    return {"lhs": lhs, "rhs": rhs, "params": params, "context": context, "dst": dst}


def run(state):
    api.mul(state["lhs"], state["rhs"], state["params"], state["context"], state["dst"])
    return state["dst"].data


def work(case):
    c = case
    size = {kind: S.DTYPE_SIZES[t] for kind, (t, _) in _TYPES.items()}
    count = c["m"] * c["k"] * size[c["lhs"]] + c["k"] * c["n"] * size[c["rhs"]] + c["m"] * c["n"] * size[c["dst"]]
    count += c["m"] * (4 * c["bias"] + 8 * c["perchannel"])
    return {"bytes": float(count), "flops": 2.0 * c["m"] * c["k"] * c["n"]}


def tolerance(case):
    # Integer results are defined exactly. fp32: four times the errors (2-norm, largest) of
    # the 32-bit sums against 64-bit ones at these depths.
    return {"rel": 4e-6, "max": 4e-5} if case["dst"] == "f32" else "exact"

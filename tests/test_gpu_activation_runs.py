"""Activations of whole runs of values (activate_run of csrc/common.hpp) in the kernels that hand results over tile by tile: every function at values of all sizes, at the lines
between its formulas and at infinities and NaN, against 64 bits."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from test_gpu_conv_ring import ACTIVATION, CODE, Layer

pytestmark = pytest.mark.gpu

NAMES = ["LINEAR", "SIGMOID", "TANH", "RELU", "SELU", "ELU", "EXPONENTIAL", "SOFTPLUS", "SOFTSIGN"]


def exact(name, v):  # (the exponential of softplus is one of 32 bits)
    with np.errstate(all="ignore"):
        return {"SIGMOID": 1.0 / (1.0 + np.exp(-v)), "TANH": np.tanh(v),
                "SELU": float(np.float32(1.05070098)) * np.where(v >= 0, v, float(np.float32(1.67326324)) * np.expm1(v)), "ELU": np.where(v >= 0, v, np.expm1(v)),
                "EXPONENTIAL": np.exp(v), "SOFTPLUS": np.where(v > 88.72, np.inf, np.log1p(np.exp(v))), "SOFTSIGN": v / (np.abs(v) + 1.0)}[name]


def values(k):
    g = h.rng(5)
    lines = [0.125, 0.0625, 87.0, 104.0, 0.3466]
    special = [0.0, -0.0, np.inf, -np.inf, np.nan, 200.0, -200.0]
    some = [s * v * f for v in lines for f in (1 - 2.0 ** -23, 1.0, 1 + 2.0 ** -22) for s in (1, -1)]
    rest = g.standard_normal(k) * 10.0 ** g.uniform(-4, 1.3, k)
    return np.concatenate([special, some, rest])[:k].astype(np.float32)


@pytest.mark.parametrize("images", [1, 90])  # small tiles; the ring kernel for 16-bit types
@pytest.mark.parametrize("filters", [448, 447])  # whole vectors; results element by element
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_every_activation(dtype, filters, images):
    layer = Layer(images, 12, 12, 256, filters, 1, 1, 1, 0)
    if filters % 4 == 0 and dtype != "f32":
        assert (cb.load_library().avhip_conv2d_ring_plan(CODE[dtype], CODE[dtype], C.byref(layer.shape), ACTIVATION, 0) >= 0) == (images > 1)
    v = values(filters)
    x, w = np.zeros(layer.x), np.zeros(layer.w)  # so that a sum is its filter's bias
    for code, name in enumerate(NAMES):
        if name in ("LINEAR", "RELU"):  # kernels of their own
            continue
        got = np.asarray(layer.forward(x, w, dtype, bias=v.astype(np.float64), activation=code), dtype=np.float64)
        assert np.array_equal(got.reshape(-1, filters), np.broadcast_to(got[0, 0, 0], (got.size // filters, filters)), equal_nan=True)
        got, want = got[0, 0, 0], exact(name, v.astype(np.float64))
        with np.errstate(all="ignore"):
            held = {"f32": want.astype(np.float32), "f16": want.astype(np.float16), "bf16": want.astype(np.float32)}[dtype].astype(np.float64)
        # the rounding of the type (half of its last place; its smallest step below that of normal values: 1 / (1 + e^-x) is 0 from e^-x = infinity on) and the function's own error, 2e-7
        half, step, own = {"f32": (2.0 ** -24, 2.0 ** -126, 4e-7), "f16": (2.0 ** -11, 2.0 ** -25, 4e-7), "bf16": (2.0 ** -8, 2.0 ** -126, 4e-7)}[dtype]
        finite = np.isfinite(held) & (np.abs(want) < {"f32": 3e38, "f16": 65000.0, "bf16": 3.3e38}[dtype])
        assert np.array_equal(np.isnan(got), np.isnan(held)), name
        assert np.all(np.abs(got - want)[finite] <= (half + own) * np.abs(want)[finite] + step), name
        odd = np.isinf(held)
        assert np.array_equal(got[odd], held[odd]), name


# where formulas made for 16-bit results are the least exact; of fp16 sigmoids only normal numbers
RANGES = [("SIGMOID", {"f16": (-9, -3), "bf16": (-87, -44)}), ("SIGMOID", {"f16": (-3, 3), "bf16": (-44, -5)}), ("TANH", (-0.3, -0.125)), ("TANH", (0.1, 0.125)),
          ("ELU", (-0.1, -0.0625)), ("SELU", (-0.1, -0.0625)), ("ELU", (-5, -1))]


@pytest.mark.parametrize("images", [1, 12])
@pytest.mark.parametrize("filters", [448, 447])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_16_bit_results_are_those_of_32_bit_functions(oracle, dtype, filters, images):
    """A function's own error cannot be seen in one 16-bit result; it shows in how many of them are rounded the other way.  An error of e of a value with p bits crosses the middle between two
    results once in 1 / (2 e 2^p) cases at most; 4e-8 is the mean error of 32-bit functions (SELU, the largest; the most seen is 6.9e-5 for fp16 and 1.1e-5 for bf16)."""
    layer = Layer(images, 12, 12, 256, filters, 1, 1, 1, 0)
    x, w = np.zeros(layer.x), np.zeros(layer.w)  # so that a sum is its filter's bias and its residual
    limit = 2 * 4e-8 * {"f16": 2.0 ** 11, "bf16": 2.0 ** 8}[dtype]
    for name, span in RANGES:
        low, high = span[dtype] if isinstance(span, dict) else span
        g = h.rng(6)
        bias = g.uniform(low / 2, high / 2, filters).astype(np.float32)
        z = h.rounded(oracle, g.uniform(low / 2, high / 2, layer.out), dtype)
        got = layer.forward(x, w, dtype, bias=bias.astype(np.float64), z=z, activation=getattr(cb, "ACTIVATION_" + name))
        want = h.rounded(oracle, exact(name, (bias + z.astype(np.float32)).astype(np.float64)), dtype)
        others = np.count_nonzero(got != want)
        assert others <= limit * want.size + 4 * np.sqrt(limit * want.size), (name, low, high, others, want.size)

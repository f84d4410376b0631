"""Tiles of 32 x 32 (csrc/conv_small.hip) of one, four and eight wavefronts, with rows of channels in whole chunks, dwords and elements, every way of handing results over; against the plain
convolution.  The plan is asked for first, so each case runs the instance that it names."""
import ctypes as C
import functools

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from test_gpu_conv_ring import ACTIVATION, CODE, ELEMENTS, VECTORS, Layer

pytestmark = pytest.mark.gpu

BAR = {"f32": 2e-6, "f16": 6e-4, "bf16": 3e-3}  # fp32 sums of up to 4500 terms (2^-24 sqrt 4500 = 4e-6 at most, a third of it typically); one rounding on store, 2^-12 and 2^-9

# wavefronts, rows of channels: arguments of Layer, one filter more gets the same tiles; 16-bit types, fp32, int8
CASES = {
    ("f16", 1, "chunks"): (7, 46, 45, 16, 132, 1, 1, 1, 0), ("f16", 4, "chunks"): (3, 44, 47, 40, 20, 3, 1, 2, 1), ("f16", 8, "chunks"): (7, 52, 51, 320, 20, 3, 2, 1, 0),
    ("f16", 1, "dwords"): (11, 35, 35, 10, 100, 1, 1, 1, 0), ("f16", 4, "dwords"): (11, 24, 25, 130, 20, 1, 1, 1, 0), ("f16", 8, "dwords"): (2, 20, 21, 318, 68, 3, 1, 1, 1),
    ("f16", 1, "elements"): (7, 57, 58, 9, 100, 1, 1, 1, 0), ("f16", 4, "elements"): (2, 56, 56, 43, 20, 3, 1, 1, 1), ("f16", 8, "elements"): (5, 21, 20, 441, 20, 3, 1, 1, 0),
    ("f32", 1, "chunks"): (11, 57, 60, 132, 20, 1, 1, 1, 0), ("f32", 4, "chunks"): (7, 29, 32, 176, 20, 1, 1, 1, 0), ("f32", 8, "chunks"): (7, 25, 24, 168, 20, 3, 1, 2, 1),
    ("f32", 1, "dwords"): (11, 58, 59, 33, 20, 1, 1, 1, 0), ("f32", 4, "dwords"): (3, 45, 48, 67, 20, 1, 1, 1, 0), ("f32", 8, "dwords"): (2, 33, 33, 205, 20, 3, 1, 1, 1),
    ("i8", 1, "chunks"): (5, 53, 53, 32, 132, 1, 1, 1, 0), ("i8", 4, "chunks"): (7, 59, 60, 688, 20, 1, 2, 1, 0), ("i8", 8, "chunks"): (2, 48, 51, 640, 20, 3, 1, 1, 1),
    ("i8", 1, "dwords"): (11, 60, 61, 8, 36, 1, 1, 1, 0), ("i8", 4, "dwords"): (3, 48, 49, 280, 20, 1, 1, 1, 0), ("i8", 8, "dwords"): (2, 54, 54, 636, 36, 3, 2, 1, 0),
    ("i8", 1, "elements"): (7, 48, 51, 9, 132, 1, 1, 1, 0), ("i8", 4, "elements"): (2, 58, 59, 81, 20, 3, 1, 2, 1), ("i8", 8, "elements"): (1, 45, 46, 347, 20, 5, 1, 1, 0),
}
FLOATS = [(dtype, waves, rows) for kind, waves, rows in CASES if kind != "i8" for dtype in (("f16", "bf16") if kind == "f16" else (kind,))]


@pytest.fixture(autouse=True)
def forced():
    lib = cb.load_library()
    lib.avhip_set_small_problem_threshold.restype = int
    previous = lib.avhip_set_small_problem_threshold(-1)
    yield
    lib.avhip_set_small_problem_threshold(previous)


def the_layer(dtype, waves, rows, filters_more=0):
    n, hh, ww, c, k, *rest = CASES["f16" if dtype == "bf16" else dtype, waves, rows]
    return Layer(n, hh, ww, c, k + filters_more, *rest)


def assert_tiles(layer, dtype, waves, hand_over):
    assert cb.load_library().avhip_conv2d_small_plan(CODE[dtype], C.byref(layer.shape), hand_over) == 32 // 2 + waves


@functools.lru_cache(maxsize=2)
def sums(dtype, waves, rows, filters_more):
    """Inputs and their plain sums, in 64 bits."""
    import torch
    from oracle import oracle as orc
    layer, g = the_layer(dtype, waves, rows, filters_more), h.rng(900 + waves)
    x = h.rounded(orc, g.standard_normal(layer.x), dtype)
    w = h.rounded(orc, g.standard_normal(layer.w) * np.sqrt(2.0 / (layer.w[1] * layer.w[2] * layer.w[3])), dtype)
    turned = w[:, ::-1, ::-1] if layer.mode else w
    xt, wt = (torch.from_numpy(np.ascontiguousarray(a)).permute(0, 3, 1, 2) for a in (x, turned))
    plain = torch.nn.functional.conv2d(xt, wt, stride=layer.stride, padding=-layer.pad, dilation=layer.dilation).permute(0, 2, 3, 1).numpy()
    return x, w, plain


@pytest.mark.parametrize("how", ["relu", "elu_residual", "relu_elements", "tanh_residual_elements"])
@pytest.mark.parametrize("case", FLOATS, ids=str)
def test_float_layers(oracle, case, how):
    dtype, waves, rows = case
    elements, act, residual = "elements" in how, how.split("_")[0].upper(), "residual" in how
    layer, g = the_layer(*case, int(elements)), h.rng(40)
    assert_tiles(layer, dtype, waves, ACTIVATION if act != "RELU" else ELEMENTS if elements else VECTORS)
    x, w, plain = sums(*case, int(elements))
    b = g.uniform(-0.1, 0.1, layer.out[3]).astype(np.float32).astype(np.float64)
    z = h.rounded(oracle, g.standard_normal(layer.out), dtype) if residual else None
    want = plain + b + (z if residual else 0.0)
    want = {"RELU": lambda v: np.maximum(v, 0.0), "ELU": lambda v: np.where(v >= 0, v, np.expm1(np.minimum(v, 0.0))), "TANH": np.tanh}[act](want)
    got = layer.forward(x, w, dtype, bias=b, z=z, activation=getattr(cb, "ACTIVATION_" + act))
    assert oracle.rel_l2(got, want) < BAR[dtype]


@pytest.mark.parametrize("filters_more", [0, 1])
@pytest.mark.parametrize("case", [case for case in CASES if case[0] == "i8"], ids=str)
def test_int8_layers(case, filters_more):
    layer, g = the_layer(*case, filters_more), h.rng(41)
    assert_tiles(layer, "i8", case[1], ELEMENTS if filters_more else VECTORS)
    x, w = g.integers(-127, 128, layer.x, dtype=np.int8), g.integers(-127, 128, layer.w, dtype=np.int8)
    b = g.integers(-2 ** 15, 2 ** 15, layer.out[3]).astype(np.int32)
    got = layer.forward(x, w, "i8", y_dtype="i32", bias=b, bias_dtype="i32")
    np.testing.assert_array_equal(got, layer.plain(x, w) + b)


@pytest.mark.parametrize("case", [case for case in FLOATS if case[2] != "chunks"], ids=str)
def test_an_infinity_stays_with_its_pixel_and_filter(case):
    """Rows of channels that end within a 16-byte chunk: what lies behind them (the next pixel, tap or filter) must not reach the sum."""
    dtype, waves, rows = case
    layer, g = the_layer(*case), h.rng(42)
    assert_tiles(layer, dtype, waves, VECTORS)
    x, w = g.standard_normal(layer.x).astype(np.float32), g.standard_normal(layer.w).astype(np.float32)
    centre = layer.w[1] // 2
    x[0, 2, 3, 0], x[1, 0, 0, 1], w[4, centre, centre, 0] = np.inf, np.nan, -np.inf  # (first channels: the pixel, tap or filter before would read them behind its last)
    got = np.isfinite(layer.forward(x, w, dtype))
    want = np.ones(layer.out, bool)
    for n, i, j in ((0, 2, 3), (1, 0, 0)):
        want[n, max(0, i - centre):i + centre + 1, max(0, j - centre):j + centre + 1] = False
    want[..., 4] = False
    assert layer.stride == 1 and np.array_equal(got, want)

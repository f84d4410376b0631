"""The implicit-GEMM kernel with a ring of LDS buffers (csrc/conv_ring.hip): every tile with every way of handing results over, at the edges of pixels, filters,
channels and stages, against the plain convolution; its operands' rows beyond the tensors count as nothing."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


class Shape(C.Structure):
    _fields_ = [(n, C.c_int) for n in "N H W C K R S Ho Wo pad_h pad_w stride_h stride_w dil_h dil_w mode".split()]


CODE = {"f16": cb.DTYPE_FLOAT16, "bf16": cb.DTYPE_BFLOAT16, "i8": cb.DTYPE_INT8, "i32": cb.DTYPE_INT32, "f32": cb.DTYPE_FLOAT32}
VECTORS, ELEMENTS, ACTIVATION = range(3)  # how results leave: HandOver of csrc/conv_small.hpp


class Layer:
    """n images of hh x ww x c, k filters of r x r, output of the input's size over the stride."""

    def __init__(self, n, hh, ww, c, k, r, stride, dilation, mode):
        self.x, self.w = (n, hh, ww, c), (k, r, r, c)
        self.pad, self.stride, self.dilation, self.mode = -(dilation * (r - 1) // 2), stride, dilation, mode
        self.out = (n, *((v - 2 * self.pad - dilation * (r - 1) - 1) // stride + 1 for v in (hh, ww)), k)
        self.shape = Shape(n, hh, ww, c, k, r, r, self.out[1], self.out[2], self.pad, self.pad, stride, stride, dilation, dilation, mode)

    def tile(self, dtype, y_dtype, hand_over, residual):
        """The tile that the call about to be made gets, or -1 where it goes to another kernel.  (Where the rule has moved, the case has to move too.)"""
        return cb.load_library().avhip_conv2d_ring_plan(CODE[dtype], CODE[y_dtype], C.byref(self.shape), hand_over, int(residual))

    def forward(self, x, w, dtype, entry="implicit_gemm", **more):
        return h.conv_forward(entry, x, w, self.out, dtype, pad=(self.pad, self.pad), stride=(self.stride, self.stride), dilation=(self.dilation, self.dilation),
                              mode=self.mode, **more)

    def plain(self, x, w):
        """The convolution on the CPU: in 64 bits for integers (exact), in 32 bits otherwise (1e-6)."""
        import torch
        kind = torch.float64 if x.dtype == np.int8 else torch.float32
        if self.mode:
            w = w[:, ::-1, ::-1]
        xt, wt = (torch.from_numpy(np.ascontiguousarray(a)).to(kind).permute(0, 3, 1, 2) for a in (x, w))
        return torch.nn.functional.conv2d(xt, wt, stride=self.stride, padding=-self.pad, dilation=self.dilation).permute(0, 2, 3, 1).double().numpy()


# tile, then the arguments of Layer: pixels and filters that fill no tile, every number of stages behind the last full round of buffers, taps that start
# inside a run of 128 bytes, rows that run over images, taps that lie apart, filters that are turned around
FLOAT_CASES = {
    "relu": [
        (0, 25, 37, 37, 32, 68, 3, 1, 1, 0), (0, 19, 42, 44, 16, 100, 1, 1, 1, 0), (0, 30, 33, 35, 144, 68, 1, 1, 1, 0), (1, 33, 23, 24, 32, 76, 3, 1, 1, 1),
        (1, 35, 23, 22, 40, 68, 3, 1, 2, 1), (1, 11, 41, 40, 48, 72, 3, 1, 2, 1), (2, 32, 26, 27, 32, 36, 3, 1, 1, 1), (2, 28, 28, 30, 16, 20, 1, 1, 1, 0),
        (2, 30, 47, 46, 160, 36, 1, 2, 1, 0), (3, 3, 37, 37, 32, 36, 3, 1, 1, 1), (3, 9, 44, 43, 16, 40, 1, 2, 1, 0), (3, 37, 15, 15, 152, 36, 1, 1, 1, 0),
    ],
    "relu_residual": [
        (0, 28, 35, 37, 40, 72, 3, 1, 2, 1), (0, 40, 36, 38, 16, 84, 1, 1, 1, 0), (0, 31, 32, 34, 72, 68, 1, 1, 1, 0), (1, 22, 34, 33, 32, 68, 3, 1, 1, 1),
        (1, 9, 44, 44, 48, 68, 3, 1, 2, 0), (1, 14, 44, 43, 40, 76, 3, 1, 2, 0), (2, 27, 27, 28, 40, 36, 3, 1, 1, 0), (2, 38, 23, 22, 24, 16, 1, 1, 1, 0),
        (2, 13, 37, 37, 80, 16, 1, 1, 1, 0), (3, 31, 17, 18, 32, 36, 3, 1, 1, 0), (3, 39, 16, 17, 16, 36, 1, 1, 1, 0), (3, 27, 27, 26, 136, 36, 1, 2, 1, 0),
    ],
    "elements": [
        (0, 31, 39, 41, 24, 66, 5, 1, 2, 1), (0, 27, 44, 44, 72, 66, 3, 1, 1, 1), (1, 19, 31, 30, 160, 65, 3, 1, 2, 0), (1, 25, 26, 28, 168, 69, 3, 1, 1, 1),
        (1, 30, 45, 47, 64, 73, 5, 2, 1, 0), (2, 17, 38, 40, 16, 33, 3, 1, 1, 0), (2, 19, 36, 35, 16, 33, 1, 1, 1, 0), (2, 27, 30, 32, 88, 33, 1, 1, 1, 0),
        (3, 25, 35, 37, 32, 37, 3, 2, 1, 0), (3, 27, 26, 28, 16, 143, 1, 2, 1, 0), (3, 25, 40, 41, 152, 33, 1, 1, 1, 0),
    ],
    "elu_residual": [
        (0, 40, 36, 36, 72, 80, 3, 1, 1, 1), (1, 21, 29, 29, 168, 68, 3, 1, 1, 1), (1, 20, 28, 30, 160, 76, 3, 1, 1, 1),
        (1, 15, 40, 42, 120, 72, 3, 1, 1, 1), (2, 14, 43, 43, 16, 36, 5, 1, 2, 1), (2, 39, 36, 37, 80, 36, 1, 1, 1, 0), (2, 31, 45, 45, 192, 36, 1, 1, 1, 0),
        (3, 12, 43, 43, 16, 44, 3, 1, 1, 0), (3, 22, 36, 37, 16, 40, 1, 1, 1, 0), (3, 19, 35, 35, 88, 36, 1, 1, 1, 0),
    ],
}
INT8_CASES = {
    "i32": [
        (0, 37, 30, 32, 64, 84, 3, 1, 2, 0), (0, 38, 46, 48, 32, 268, 1, 2, 1, 0), (1, 29, 24, 24, 80, 80, 3, 1, 2, 1), (1, 34, 21, 23, 96, 76, 3, 1, 1, 0),
        (2, 26, 27, 27, 64, 16, 3, 1, 1, 0), (2, 39, 24, 24, 32, 148, 1, 2, 1, 0), (3, 39, 19, 21, 64, 36, 3, 2, 1, 0), (3, 19, 23, 23, 32, 72, 1, 2, 1, 0),
    ],
    "i32_elements": [
        (0, 36, 42, 41, 48, 66, 5, 1, 1, 0), (1, 13, 37, 37, 336, 70, 3, 1, 1, 0), (2, 34, 43, 44, 48, 15, 3, 2, 2, 1), (3, 37, 14, 16, 64, 38, 3, 1, 1, 1),
    ],
    "requantised": [
        (0, 37, 30, 32, 64, 84, 3, 1, 2, 0), (0, 31, 42, 42, 32, 68, 1, 1, 1, 0), (1, 9, 45, 45, 64, 76, 3, 1, 1, 1), (1, 29, 24, 24, 80, 80, 3, 1, 2, 1),
        (2, 26, 27, 27, 64, 16, 3, 1, 1, 0), (2, 5, 46, 48, 32, 68, 1, 1, 1, 0), (3, 39, 19, 21, 64, 36, 3, 2, 1, 0), (3, 19, 23, 23, 32, 72, 1, 2, 1, 0),
    ],
    "requantised_elements": [
        (0, 29, 43, 42, 112, 87, 3, 1, 1, 0), (1, 13, 37, 37, 336, 70, 3, 1, 1, 0), (2, 34, 43, 44, 48, 15, 3, 2, 2, 1), (3, 37, 14, 16, 64, 38, 3, 1, 1, 1),
    ],
    "f32_residual": [
        (0, 23, 42, 43, 64, 76, 3, 1, 1, 0), (1, 16, 43, 44, 64, 68, 3, 1, 1, 0), (2, 39, 23, 24, 64, 16, 3, 1, 1, 0), (3, 17, 24, 25, 64, 16, 3, 1, 2, 0),
    ],
    "f32_elu": [
        (0, 30, 44, 45, 144, 68, 3, 1, 1, 0), (1, 9, 44, 45, 320, 68, 3, 1, 1, 0), (2, 32, 30, 29, 96, 16, 3, 1, 1, 0), (3, 20, 33, 34, 32, 44, 3, 1, 1, 1),
    ],
}

ids = lambda c: c[0] + "-" + "-".join(map(str, c[1]))
listed = lambda cases: [(how, c) for how in cases for c in cases[how]]


@pytest.mark.parametrize("case", listed(FLOAT_CASES), ids=ids)
def test_float_layers(case):
    how, (tile, *rest) = case
    layer, residual = Layer(*rest), "residual" in how
    n, k, r, c = layer.x[0], *layer.w[:2], layer.w[3]
    dtype = "bf16" if (n + k // 4) % 2 else "f16"
    assert layer.tile(dtype, dtype, VECTORS if how.startswith("relu") else ELEMENTS if how == "elements" else ACTIVATION, residual) == tile
    g = h.rng(100 + n)
    x = orc.round_to(g.standard_normal(layer.x), dtype)
    w = orc.round_to(g.standard_normal(layer.w) * np.sqrt(2.0 / (r * r * c)), dtype)
    b = g.uniform(-0.1, 0.1, k).astype(np.float32).astype(np.float64)
    z = orc.round_to(g.standard_normal(layer.out), dtype) if residual else None
    elu = how.startswith("elu")
    got = layer.forward(x, w, dtype, bias=b, z=z, activation=cb.ACTIVATION_ELU if elu else cb.ACTIVATION_RELU)
    want = layer.plain(x.astype(np.float32), w.astype(np.float32)) + b
    if residual:
        want = want + z
    want = np.where(want > 0, want, np.expm1(np.minimum(want, 0)) if elu else 0)
    # one rounding of the result: 2^-8 (bf16) and 2^-11 (fp16) of a value at most, some 0.4 of that in the mean of squares
    assert orc.rel_l2(got, want) < (2e-3 if dtype == "bf16" else 3e-4)


@pytest.mark.parametrize("case", listed(INT8_CASES), ids=ids)
def test_int8_layers(case):
    how, (tile, *rest) = case
    layer, residual = Layer(*rest), "residual" in how
    n, k, r, c = layer.x[0], *layer.w[:2], layer.w[3]
    y_dtype = "i8" if how.startswith("requantised") else "f32" if how.startswith("f32") else "i32"
    assert layer.tile("i8", y_dtype, ELEMENTS if "elements" in how else ACTIVATION if "elu" in how else VECTORS, residual) == tile
    g = h.rng(200 + n)
    x = g.integers(-127, 128, layer.x, dtype=np.int8)
    w = g.integers(-127, 128, layer.w, dtype=np.int8)
    sums = layer.plain(x, w)
    if y_dtype == "f32":
        b = g.uniform(-0.1, 0.1, k).astype(np.float32)
        z = g.standard_normal(layer.out).astype(np.float32) if residual else None
        got = layer.forward(x, w, "i8", y_dtype="f32", bias=b, bias_dtype="f32", z=z, alpha1=1e-5, activation=cb.ACTIVATION_RELU if residual else cb.ACTIVATION_ELU)
        want = float(np.float32(1e-5)) * sums + b + (z if residual else 0)
        want = np.maximum(want, 0) if residual else np.where(want > 0, want, np.expm1(np.minimum(want, 0)))
        assert orc.rel_l2(got, want) < 1e-6  # a few roundings of 2^-24
        return
    b = g.integers(-2 ** 15, 2 ** 15, k).astype(np.int32)
    if y_dtype == "i32":
        got = layer.forward(x, w, "i8", y_dtype="i32", bias=b, bias_dtype="i32")
        assert np.array_equal(got.astype(np.int64), (sums + b).astype(np.int64))
        return
    scale = g.uniform(1e-5, 4e-4, k).astype(np.float32)
    got = layer.forward(x, w, "i8", entry="requant", bias=b, bias_dtype="i32", scale=scale, activation=cb.ACTIVATION_RELU)
    # one rounding of the product, one to an integer
    want = np.rint(np.maximum(sums + b, 0).astype(np.float32) * scale)
    assert np.array_equal(got.astype(np.int64), np.clip(want, -128, 127).astype(np.int64))


@pytest.mark.parametrize("hand_over", [VECTORS, ELEMENTS], ids=["vectors", "elements"])
@pytest.mark.parametrize("tile", range(4))
def test_nothing_behind_the_tensors_counts(tile, hand_over):
    """Infinities and NaN in the pixels next to a tap's image border and in the filters' neighbours reach no other output."""
    rest = next(c[1:] for c in FLOAT_CASES["relu" if hand_over == VECTORS else "elements"] if c[0] == tile and c[5] > 1)
    layer = Layer(*rest)
    assert layer.tile("f16", "f16", hand_over, False) == tile
    n, hh, ww, c = layer.x
    k, r = layer.w[:2]
    g = h.rng(7)
    x = orc.round_to(g.standard_normal(layer.x), "f16")
    w = orc.round_to(g.standard_normal(layer.w) * 0.05, "f16")
    x[0, 0, 0, 3], x[1, hh - 1, ww - 1, 0], x[n - 1, hh - 1, ww - 1, c - 1] = np.inf, np.nan, np.inf
    w[k - 2, r // 2, r // 2, 2], w[k - 1, r // 2, r // 2, c - 1] = np.nan, np.inf  # (the tap that never meets the border)
    got = layer.forward(x, w, "f16")
    want = layer.plain(x.astype(np.float32), w.astype(np.float32))
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    assert orc.rel_l2(got[finite], want[finite]) < 3e-4

"""The implicit-GEMM kernel with a ring of LDS buffers (csrc/conv_ring.hip): every tile, at the edges of pixels, filters, channels
and stages, against the oracle; its operands' rows beyond the tensors count as nothing."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


class Shape(C.Structure):
    _fields_ = [(n, C.c_int) for n in "N H W C K R S Ho Wo pad_h pad_w stride_h stride_w dil_h dil_w mode".split()]


def plan_of(n, h_, w_, c, k, r, stride, dtype, y_dtype):
    out = [(v + 2 * (r // 2) - r) // stride + 1 for v in (h_, w_)]
    s = Shape(n, h_, w_, c, k, r, r, out[0], out[1], -(r // 2), -(r // 2), stride, stride, 1, 1, 0)
    code = {"f16": cb.DTYPE_FLOAT16, "bf16": cb.DTYPE_BFLOAT16, "i8": cb.DTYPE_INT8, "i32": cb.DTYPE_INT32}
    return cb.load_library().avhip_conv2d_ring_plan(code[dtype], code[y_dtype], C.byref(s)), out


def torch_conv(x, w, r, stride):
    """The plain convolution on the CPU: in 64 bits for integers (exact), in 32 bits otherwise (1e-6)."""
    import torch
    kind = torch.float64 if x.dtype == np.int8 else torch.float32
    xt, wt = (torch.from_numpy(np.ascontiguousarray(a)).to(kind).permute(0, 3, 1, 2) for a in (x, w))
    return torch.nn.functional.conv2d(xt, wt, stride=stride, padding=r // 2).permute(0, 2, 3, 1).double().numpy()


# tile, n, h, w, c, k, r, stride: pixels and filters that fill no tile, every number of stages behind the last full round of buffers, one stage alone,
# taps that start inside a run of 128 bytes, rows that run over images
FLOAT_CASES = [
    (0, 21, 42, 44, 16, 80, 1, 1), (0, 31, 21, 21, 72, 260, 1, 1), (0, 22, 39, 41, 16, 68, 3, 1), (0, 30, 26, 28, 32, 140, 3, 1),
    (1, 23, 36, 36, 24, 68, 3, 1), (1, 35, 47, 46, 32, 80, 3, 2), (1, 36, 42, 43, 352, 68, 1, 2), (1, 34, 21, 23, 48, 76, 3, 1),
    (2, 9, 43, 43, 16, 28, 1, 1), (2, 29, 36, 36, 136, 72, 1, 2), (2, 28, 28, 29, 32, 20, 3, 1), (2, 27, 25, 27, 16, 24, 5, 1),
    (3, 23, 43, 42, 16, 20, 1, 2), (3, 6, 27, 26, 16, 40, 3, 1), (3, 19, 29, 31, 24, 44, 3, 2), (3, 6, 15, 16, 16, 164, 5, 1), (3, 15, 25, 27, 32, 68, 3, 2),
]
INT8_CASES = [(0, 15, 40, 42, 32, 132, 3, 1), (1, 14, 44, 46, 48, 412, 3, 2), (2, 37, 22, 21, 32, 24, 3, 1), (2, 39, 30, 30, 32, 80, 1, 2), (3, 38, 6, 7, 48, 548, 3, 2),
              (3, 25, 29, 30, 144, 36, 1, 2)]
ids = lambda c: "-".join(map(str, c))


@pytest.mark.parametrize("how", ["relu", "elements", "elu_residual"])
@pytest.mark.parametrize("case", FLOAT_CASES, ids=ids)
def test_float_layers(case, how):
    tile, n, hh, ww, c, k, r, stride = case
    dtype = "bf16" if (n + k // 4) % 2 else "f16"
    plan, out = plan_of(n, hh, ww, c, k, r, stride, dtype, dtype)
    # (where the rule has moved, the case has to move too)
    assert plan == tile
    if how == "elements":
        k -= 1
    g = h.rng(100 + n)
    x = orc.round_to(g.standard_normal((n, hh, ww, c)), dtype)
    w = orc.round_to(g.standard_normal((k, r, r, c)) * np.sqrt(2.0 / (r * r * c)), dtype)
    b = g.uniform(-0.1, 0.1, k).astype(np.float32).astype(np.float64)
    z = orc.round_to(g.standard_normal((n, out[0], out[1], k)), dtype) if how == "elu_residual" else None
    got = h.conv_forward("implicit_gemm", x, w, (n, out[0], out[1], k), dtype, bias=b, z=z,
                         activation=cb.ACTIVATION_ELU if z is not None else cb.ACTIVATION_RELU, pad=(-(r // 2), -(r // 2)), stride=(stride, stride))
    want = torch_conv(x.astype(np.float32), w.astype(np.float32), r, stride) + b
    if z is not None:
        want = want + z
        want = np.where(want > 0, want, np.expm1(np.minimum(want, 0)))
    else:
        want = np.maximum(want, 0)
    # one rounding of the result: 2^-9 (bf16) and 2^-12 (fp16) at most, half of that on average
    assert orc.rel_l2(got, want) < (2e-3 if dtype == "bf16" else 3e-4)


@pytest.mark.parametrize("case", INT8_CASES, ids=ids)
def test_int8_layers(case):
    tile, n, hh, ww, c, k, r, stride = case
    plan, out = plan_of(n, hh, ww, c, k, r, stride, "i8", "i32")
    assert plan == tile
    g = h.rng(200 + n)
    x = g.integers(-127, 128, (n, hh, ww, c), dtype=np.int8)
    w = g.integers(-127, 128, (k, r, r, c), dtype=np.int8)
    b = g.integers(-2 ** 15, 2 ** 15, k).astype(np.int32)
    got = h.conv_forward("implicit_gemm", x, w, (n, out[0], out[1], k), "i8", y_dtype="i32", bias=b, bias_dtype="i32", pad=(-(r // 2), -(r // 2)),
                         stride=(stride, stride))
    want = torch_conv(x, w, r, stride) + b
    assert np.array_equal(got.astype(np.int64), want.astype(np.int64))


def test_nothing_behind_the_tensors_counts():
    """Infinities and NaN in the pixels next to a tap's image border and in the filters' neighbours reach no other output."""
    n, hh, ww, c, k, r, stride = 6, 27, 26, 16, 40, 3, 1
    assert plan_of(n, hh, ww, c, k, r, stride, "f16", "f16")[0] == 3
    g = h.rng(7)
    x = orc.round_to(g.standard_normal((n, hh, ww, c)), "f16")
    w = orc.round_to(g.standard_normal((k, r, r, c)) * 0.1, "f16")
    x[2, 0, 0, 3], x[3, 26, 25, 0] = np.inf, np.nan
    w[17, 1, 1, 2] = np.nan
    got = h.conv_forward("implicit_gemm", x, w, (n, hh, ww, k), "f16")
    want = torch_conv(x.astype(np.float32), w.astype(np.float32), r, stride)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))

"""Tiles of 16 x 16 (csrc/conv_small16.hip) against the oracle: one tile and many, ragged both ways, one wavefront to eight of them, shares of k from less than a stage to several rounds,
borders, strides, dilations, flipped filters, every hand-over of results.  The plan is asked for first, for few channels that which stands before the kernels made for them, so each case runs
the instance that it names."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h

pytestmark = pytest.mark.gpu

SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1}
BAR = {"f32": 2e-6, "f16": 6e-4, "bf16": 3e-3}  # fp32 sums of up to 4096 terms (2^-24 sqrt 4096 = 4e-6 at most, a third of it typically); one rounding on store, 2^-12 and 2^-9


class Shape(C.Structure):
    _fields_ = [(n, C.c_int) for n in "N H W C K R S Ho Wo pad_h pad_w stride_h stride_w dil_h dil_w mode".split()]


# wavefronts; images, rows, columns, 16-byte chunks of channels; filters, their rows and columns; the rest of the geometry
CASES = [(1, (1, 5, 5, 8), (16, 1, 1), {}),                                                             # one stage, a second tile of nine pixels
         (1, (7, 9, 11, 2), (44, 1, 1), dict(stride=(2, 2))),                                           # two chunks
         (1, (20, 16, 16, 16), (96, 1, 1), {}),                                                         # 1920 tiles
         (4, (25, 9, 7, 8), (36, 3, 3), dict(pad=(-1, -1))),                                             # the last tile ragged either way
         (4, (3, 20, 17, 6), (100, 3, 3), dict(pad=(-1, -1))),
         (4, (25, 13, 11, 4), (64, 3, 5), dict(pad=(-2, -4), stride=(2, 1), dilation=(2, 2), mode=1)),
         (8, (1, 4, 4, 13), (4, 5, 5), dict(pad=(-2, -2))),                                             # one tile; the last wavefronts have less to do, or nothing
         (8, (2, 6, 5, 16), (17, 4, 8), dict(pad=(-3, -7)))]                                            # 32 taps, several rounds of two stages


@pytest.fixture(autouse=True)
def forced():
    lib = cb.load_library()
    lib.avhip_set_small_problem_threshold.restype = int
    previous = lib.avhip_set_small_problem_threshold(-1)
    yield
    lib.avhip_set_small_problem_threshold(previous)


@pytest.mark.parametrize("act, z", [("RELU", False), ("LINEAR", True), ("ELU", True)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "i8"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_the_oracle(oracle, case, dtype, act, z):
    waves, (N, H, W, chunks), (K, R, S), geometry = CASES[case]
    Cin = chunks * 16 // SIZE[dtype]
    (ph, pw), (sh, sw), (dh, dw) = geometry.get("pad", (0, 0)), geometry.get("stride", (1, 1)), geometry.get("dilation", (1, 1))
    ys = (N, (H - 2 * ph - ((R - 1) * dh + 1)) // sh + 1, (W - 2 * pw - ((S - 1) * dw + 1)) // sw + 1, K)
    shape = Shape(N, H, W, Cin, K, R, S, ys[1], ys[2], ph, pw, sh, sw, dh, dw, geometry.get("mode", 0))
    code = {"f32": cb.DTYPE_FLOAT32, "f16": cb.DTYPE_FLOAT16, "bf16": cb.DTYPE_BFLOAT16, "i8": cb.DTYPE_INT8}[dtype]
    assert cb.load_library().avhip_conv2d_small_plan(code, C.byref(shape), 0) == 16 // 2 + waves
    geometry = {"pad": (0, 0), **geometry}
    g = h.rng(700 + case)
    if dtype == "i8":
        if act != "RELU":
            pytest.skip("integer sums: one hand-over of whole vectors, one element by element, both with the filters of these cases")
        x, w = g.integers(-127, 128, (N, H, W, Cin), dtype=np.int8), g.integers(-127, 128, (K, R, S, Cin), dtype=np.int8)
        b = g.integers(-2 ** 15, 2 ** 15, K).astype(np.int32)
        got = h.conv_forward("implicit_gemm", x, w, ys, "i8", y_dtype="i32", bias=b, bias_dtype="i32", **geometry)
        np.testing.assert_array_equal(got, oracle.conv2d_i8(x, w, b, **geometry))
        return
    x = h.rounded(oracle, g.standard_normal((N, H, W, Cin)), dtype)
    w = h.rounded(oracle, g.standard_normal((K, R, S, Cin)) * np.sqrt(2.0 / (R * S * Cin)), dtype)
    b = g.uniform(-0.1, 0.1, K).astype(np.float32).astype(np.float64)
    res = h.rounded(oracle, g.standard_normal(ys), dtype) if z else None
    code = getattr(cb, "ACTIVATION_" + act)
    got = h.conv_forward("implicit_gemm", x, w, ys, dtype, bias=b, z=res, activation=code, **geometry)
    assert oracle.rel_l2(got, oracle.conv2d(x, w, b, res, activation=code, **geometry)) < BAR[dtype]


# wavefronts; images, rows, columns, channels of each type (absent: no such row); filters, their rows and columns; the rest of the geometry.  Rows of channels that are no whole chunks
# (dwords, elements), that are one chunk, that are less than one
ROWS = [(1, (3, 7, 5), dict(f32=9, f16=18, bf16=1, i8=36), (18, 1, 1), {}), (8, (2, 9, 7), dict(f32=33, f16=66, bf16=65, i8=131), (20, 3, 3), dict(pad=(-1, -1))),
        (8, (1, 5, 4), dict(f32=101, f16=201, bf16=203, i8=403), (33, 3, 5), dict(pad=(-1, -2), stride=(2, 1))), (1, (3, 8, 9), dict(f32=4, f16=8, bf16=8, i8=16), (40, 1, 1), {}),
        (1, (20, 12, 9), dict(f32=4, f16=8, bf16=2, i8=16), (36, 3, 3), dict(pad=(-1, -1))), (1, (20, 12, 9), dict(f32=3, f16=3, bf16=4, i8=5), (64, 3, 3), dict(pad=(-1, -1), mode=1)),
        (4, (9, 13, 12), dict(f32=2, f16=3, bf16=3, i8=3), (32, 5, 5), dict(pad=(-2, -2), stride=(2, 2)))]


@pytest.mark.parametrize("act", ["RELU", "ELU"])  # few channels: RELU by estimate, before the kernels made for them; ELU as any layer
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "i8"])
@pytest.mark.parametrize("case", range(len(ROWS)))
def test_rows_of_channels(oracle, case, dtype, act):
    waves, (N, H, W), channels, (K, R, S), geometry = ROWS[case]
    Cin = channels[dtype]
    lib = cb.load_library()
    if act == "RELU":  # (of int8, whose sums have no activation here, the half by estimate)
        lib.avhip_set_small_problem_threshold(4096)
    (ph, pw), (sh, sw) = geometry.get("pad", (0, 0)), geometry.get("stride", (1, 1))
    ys = (N, (H - 2 * ph - R) // sh + 1, (W - 2 * pw - S) // sw + 1, K)
    shape = Shape(N, H, W, Cin, K, R, S, ys[1], ys[2], ph, pw, sh, sw, 1, 1, geometry.get("mode", 0))
    code = {"f32": cb.DTYPE_FLOAT32, "f16": cb.DTYPE_FLOAT16, "bf16": cb.DTYPE_BFLOAT16, "i8": cb.DTYPE_INT8}[dtype]
    query = lib.avhip_conv2d_plain_small_plan if act == "RELU" and K % 4 == 0 else lib.avhip_conv2d_small_plan  # (single filters: no kernel for few channels takes them)
    arguments = (code, C.byref(shape)) if query is lib.avhip_conv2d_plain_small_plan else (code, C.byref(shape), 2 if act == "ELU" and dtype != "i8" else 1 if K % 4 else 0)
    assert query(*arguments) in [8 + n for n in ((1, 4, 8) if waves == 4 else (waves,))]
    geometry = {"pad": (0, 0), **geometry}
    g = h.rng(800 + case)
    if dtype == "i8":
        x, w = g.integers(-127, 128, (N, H, W, Cin), dtype=np.int8), g.integers(-127, 128, (K, R, S, Cin), dtype=np.int8)
        b = g.integers(-2 ** 15, 2 ** 15, K).astype(np.int32)
        got = h.conv_forward("implicit_gemm", x, w, ys, "i8", y_dtype="i32", bias=b, bias_dtype="i32", **geometry)
        np.testing.assert_array_equal(got, oracle.conv2d_i8(x, w, b, **geometry))
        return
    x = h.rounded(oracle, g.standard_normal((N, H, W, Cin)), dtype)
    w = h.rounded(oracle, g.standard_normal((K, R, S, Cin)) * np.sqrt(2.0 / (R * S * Cin)), dtype)
    b = g.uniform(-0.1, 0.1, K).astype(np.float32).astype(np.float64)
    code = getattr(cb, "ACTIVATION_" + act)
    got = h.conv_forward("implicit_gemm", x, w, ys, dtype, bias=b, activation=code, **geometry)
    assert oracle.rel_l2(got, oracle.conv2d(x, w, b, activation=code, **geometry)) < BAR[dtype]


def test_an_infinity_stays_with_its_pixel_and_filter():
    """Pixels outside the image, filters past the last and shares of k past the end count as zeros, whatever lies behind the tensors."""
    x, w = np.ones((1, 5, 5, 32), np.float32), np.ones((18, 3, 3, 32), np.float32)
    x[0, 0, 0, 3], w[7] = np.inf, np.nan
    finite = np.isfinite(h.conv_forward("implicit_gemm", x, w, (1, 5, 5, 18), "f16"))
    want = np.ones((1, 5, 5, 18), bool)
    want[0, :2, :2] = want[..., 7] = False
    assert np.array_equal(finite, want)

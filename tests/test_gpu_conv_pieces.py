"""fp32 convolutions whose products are of bf16 pieces (gather kernel, 64 x 64 small tiles): no less precise than fp32 products, and the same answers where
values have no such pieces."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from test_gpu_winograd import ConvShape

pytestmark = pytest.mark.gpu


def torch_conv(x, w, stride):
    import torch
    xt, wt = (torch.from_numpy(a.astype(np.float64)).permute(0, 3, 1, 2) for a in (x, w))
    return torch.nn.functional.conv2d(xt, wt, stride=stride, padding=w.shape[1] // 2).permute(0, 2, 3, 1).numpy()


# n, h, w, c, k, r: k stages that divide by no number of wavefronts, pixels and filters that fill no tile.  Small tiles of 64 x 64 (the last: channels in
# dwords, not in whole chunks), and the gather kernel, which is what is left for layers with a stride where small tiles are switched off.
SMALL = [(11, 37, 37, 36, 200, 3), (12, 52, 40, 84, 100, 3), (12, 33, 38, 50, 196, 3)]
GATHER = [(12, 37, 35, 64, 132, 3), (7, 41, 44, 36, 200, 5)]
CASES = [("small",) + c for c in SMALL] + [("gather",) + c for c in GATHER]


@pytest.fixture
def kernel(case):
    """The kernel that the case is for takes it."""
    which, n, hh, ww, c, k, r = case
    lib = cb.load_library()
    lib.avhip_set_small_problem_threshold.restype = int
    previous = lib.avhip_set_small_problem_threshold(4096 if which == "small" else 0)
    shape = ConvShape(n, hh, ww, c, k, r, r, (hh - 1) // 2 + 1, (ww - 1) // 2 + 1, -(r // 2), -(r // 2), 2, 2, 1, 1, 0)
    assert lib.avhip_conv2d_small_plan(cb.DTYPE_FLOAT32, C.byref(shape), 0) == (2 * 16 + 4 if which == "small" else 0)
    assert which == "small" or c % 4 == 0, "the branch-free loaders of the gather kernel"
    yield
    lib.avhip_set_small_problem_threshold(previous)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -50])
def test_error_of_a_32_bit_sum(kernel, case, scale):
    _, n, hh, ww, c, k, r = case
    g = h.rng(50 + c)
    x = (g.standard_normal((n, hh, ww, c)) * scale).astype(np.float32)
    w = (g.standard_normal((k, r, r, c)) * np.sqrt(2.0 / (r * r * c))).astype(np.float32)
    want = torch_conv(x, w, 2)
    got = h.conv_forward("implicit_gemm", x, w, want.shape, "f32", pad=(-(r // 2), -(r // 2)), stride=(2, 2))
    # at most sqrt(k) roundings of 2^-24 as they add up at random (fp32 products: 2e-7 to 6e-7)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < np.sqrt(r * r * c) * 2.0 ** -24


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_values_without_pieces(kernel, case):
    _, n, hh, ww, c, k, r = case
    g = h.rng(60 + c)
    x = g.standard_normal((n, hh, ww, c)).astype(np.float32)
    w = (g.standard_normal((k, r, r, c)) * 0.05).astype(np.float32)
    x[1, 0, 0, 3], x[2, 9, 9, 0], x[3, 30, 31, c - 1], x[4, 5, 6, 1] = np.inf, np.nan, -np.inf, np.finfo(np.float32).max
    want = torch_conv(x, w, 2)
    got = h.conv_forward("implicit_gemm", x, w, want.shape, "f32", pad=(-(r // 2), -(r // 2)), stride=(2, 2))
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    large = np.abs(want) > 1e30
    ordinary, large = finite & ~large, finite & large
    assert np.linalg.norm(got[ordinary] - want[ordinary]) / np.linalg.norm(want[ordinary]) < 1e-6
    assert large.any() and (np.abs(got[large] - want[large]) <= 1e-6 * np.abs(want[large])).all()

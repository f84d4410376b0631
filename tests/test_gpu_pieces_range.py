"""fp32 products of bf16 pieces (struct Pieces of csrc/mfma_core.hpp): operands of any size, down to the subnormal numbers, are no less precise than in fp32
products.  One case for each kernel that has them; the one-kernel F(4x4, 3x3) has its own in test_gpu_f4_pieces.py."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from test_gpu_winograd import ConvShape

pytestmark = pytest.mark.gpu

# (operands' exponents: the second piece of the smaller one is below bf16's subnormal numbers from 2^-118 on, the first from 2^-134 on; the last but one
# has sums that are infinite with the scale of the pieces, the last an operand)
SCALES = [(0, 0), (-112, 8), (-118, 8), (8, -118), (-124, 20), (-138, 40), (40, -138), (60, 50), (122, -60)]


def operands(shapes, scales):
    g = h.rng(80)
    return [(g.standard_normal(s) * 2.0 ** e).astype(np.float32) for s, e in zip(shapes, scales)]


def check(got, want, k):
    """At most a rounding of 2^-24 for each of the k products as they add up at random."""
    assert np.linalg.norm(got.astype(np.float64) - want) < np.sqrt(k) * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("scales", SCALES)
def test_tn_product(scales):
    """Tiles of 64 x 64."""
    assert cb.load_library().avhip_gemm_tn_side(4, 130, 64, 60, 200) == 64
    A, B = operands([(130, 200, 64), (130, 200, 60)], scales)
    got = h.gemm(A, B, np.zeros((130, 64, 60), np.float32), "f32", True, False, batched=True)
    check(got, np.matmul(A.astype(np.float64).transpose(0, 2, 1), B.astype(np.float64)), 200)


@pytest.mark.parametrize("batch, K", [(600, 100), (3, 260)])
@pytest.mark.parametrize("scales", SCALES)
def test_nt_product(scales, batch, K):
    """The one-tile kernel: 65 to 128 of k and 600 tiles, or more of k."""
    A, B = operands([(batch, 33, K), (batch, 64, K)], scales)
    got = h.gemm(A, B, np.zeros((batch, 33, 64), np.float32), "f32", False, True, batched=True)
    check(got, np.matmul(A.astype(np.float64), B.astype(np.float64).transpose(0, 2, 1)), K)


def torch_conv(x, w):
    import torch
    xt, wt = (torch.from_numpy(a.astype(np.float64)).permute(0, 3, 1, 2) for a in (x, w))
    return torch.nn.functional.conv2d(xt, wt, stride=2, padding=1).permute(0, 2, 3, 1).numpy()


# the gather kernel; the same with k in parts through the workspace; small tiles of 64 x 64, rows in whole chunks and in dwords
@pytest.mark.parametrize("entry, threshold, case", [("implicit_gemm", 0, (9, 17, 15, 36, 132)), ("dispatch", 0, (4, 14, 14, 512, 132)),
                                                    ("implicit_gemm", 4096, (15, 43, 29, 36, 132)), ("implicit_gemm", 4096, (12, 33, 38, 50, 196))],
                         ids=["gather", "parts", "small_chunks", "small_dwords"])
@pytest.mark.parametrize("scales", SCALES)
def test_convolution(scales, entry, threshold, case):
    n, hh, ww, c, k = case
    x, w = operands([(n, hh, ww, c), (k, 3, 3, c)], scales)
    want = torch_conv(x, w)
    shape = ConvShape(n, hh, ww, c, k, 3, 3, want.shape[1], want.shape[2], -1, -1, 2, 2, 1, 1, 0)
    lib = cb.load_library()
    lib.avhip_set_small_problem_threshold.restype = int
    previous = lib.avhip_set_small_problem_threshold(threshold)
    try:
        assert lib.avhip_conv2d_small_plan(cb.DTYPE_FLOAT32, C.byref(shape), 0) == (2 * 16 + 4 if threshold else 0)
        parts = C.c_int64(0)
        assert lib.avhip_conv2d_split_k_workspace(cb.DTYPE_FLOAT32, C.byref(shape), C.byref(parts)) == 0 and (parts.value > 0) == (entry == "dispatch")
        got = h.conv_forward(entry, x, w, want.shape, "f32", stride=(2, 2))
    finally:
        lib.avhip_set_small_problem_threshold(previous)
    check(got, want, 9 * c)

"""fp32 3x3 layers that the dispatcher takes to direct sums and not to the fused Winograd kernel (csrc/backend.cpp, direct_before_fused): its result is the implicit GEMM's in
every bit, and has the error of direct sums."""
import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# images, rows, columns, channels, filters, activation, residual: full rounds of the fused kernel's workgroups, hardly begun ones, filters that fill no block, rows in no whole vectors, channels in no whole chunks (which the fused kernel declines)
CASES = [(246, 13, 13, 32, 32, "relu", False), (64, 29, 29, 64, 48, "relu", False), (34, 40, 43, 32, 33, "linear", True), (45, 48, 51, 32, 32, "sigmoid", True),
         (22, 36, 35, 96, 55, "elu", False), (11, 39, 39, 96, 192, "tanh", False), (42, 31, 31, 60, 99, "relu", True), (42, 31, 31, 61, 99, "linear", False)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_direct_sums(case):
    n, hh, ww, c, k, act, residual = case
    g = h.rng(n + k)
    x = g.standard_normal((n, hh, ww, c)).astype(np.float32).astype(np.float64)
    w = (g.standard_normal((k, 3, 3, c)) * np.sqrt(2.0 / (9 * c))).astype(np.float32).astype(np.float64)
    b = g.uniform(-0.1, 0.1, k).astype(np.float32).astype(np.float64)
    shape = (n, hh, ww, k)
    z = g.standard_normal(shape).astype(np.float32).astype(np.float64) if residual else None
    more = dict(bias=b, z=z, activation=getattr(cb, "ACTIVATION_" + act.upper()))
    got = h.conv_forward("dispatch", x, w, shape, "f32", **more)
    assert np.array_equal(got, h.conv_forward("implicit_gemm", x, w, shape, "f32", **more))
    some = slice(0, 2)  # the whole batch has been compared above; the oracle is slow
    want = orc.conv2d(x[some], w, b, z=z[some] if residual else None, activation=getattr(orc, act.upper()))
    assert orc.rel_l2(got[some], want) < 1e-6  # direct sums 1.2e-7 to 4.3e-7 (a k of one wavefront the most), the fused kernel 1.7e-7 to 2.7e-7

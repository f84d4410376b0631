"""The A B^T product of csrc/gemm.hip in fp32 with k of 65 to 128 on both sides of the line (600 tiles of 128 x 128) from which it is made of
bf16 pieces: against 64 bits, and where values have no such pieces."""
import numpy as np
import pytest

import helpers as h

pytestmark = pytest.mark.gpu


def product(A, B):
    return np.matmul(A, B.transpose(0, 2, 1))


@pytest.mark.parametrize("alpha,beta", [(None, None), (1.5, 0.5)])
@pytest.mark.parametrize("shape", [(600, 33, 64, 68), (599, 33, 64, 68), (150, 257, 132, 128), (300, 130, 20, 96), (101, 129, 260, 100)])
def test_short_fp32_products(shape, alpha, beta):
    """At most sqrt(K) roundings of 2^-24 as they add up at random, with a factor of two, and one more of the result with alpha and beta."""
    batch, M, N, K = shape
    g = h.rng(41)
    A, B, C0 = (g.standard_normal(s).astype(np.float32) for s in ((batch, M, K), (batch, N, K), (batch, M, N)))
    got = h.gemm(A, B, C0, "f32", False, True, alpha, beta, batched=True)
    want = (alpha or 1.0) * product(A.astype(np.float64), B.astype(np.float64)) + (beta or 0.0) * C0
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2 * np.sqrt(K + 1) * 2.0 ** -24


def test_short_fp32_values_without_pieces():
    batch, M, N, K = 600, 64, 64, 128
    g = h.rng(42)
    A, B = (g.standard_normal((batch, n, K)).astype(np.float32) for n in (M, N))
    A[3, 7, 5], A[4, 50, 127], B[5, 0, 0], A[6, 20, 20] = np.inf, np.nan, -np.inf, np.finfo(np.float32).max
    B[6, :, 20] *= 1e-3
    with np.errstate(invalid="ignore", over="ignore"):
        want = product(A.astype(np.float64), B.astype(np.float64))
    got = h.gemm(A, B, np.zeros((batch, M, N), np.float32), "f32", False, True, batched=True)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    rows = np.abs(want).max(axis=2, keepdims=True, where=finite, initial=1.0)
    assert (np.abs(got[finite] - want[finite]) <= 2e-5 * np.broadcast_to(rows, want.shape)[finite]).all()

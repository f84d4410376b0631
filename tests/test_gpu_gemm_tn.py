"""The A^T B product of the weight gradient (csrc/gemm_tn.hip): fp32 through three bf16 pieces a value, against 64 bits and where values
have no such pieces; 16-bit pairs in tiles of 32 x 32."""
import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h

pytestmark = pytest.mark.gpu


def product(A, B):
    return np.matmul(A.transpose(0, 2, 1), B)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -60, 2.0 ** 55])
@pytest.mark.parametrize("shape", [(130, 64, 64, 130), (36, 128, 97, 1031), (33, 100, 126, 17)])
def test_fp32_pieces_are_no_less_precise(shape, scale):
    """Tiles of 64 x 64.  What is dropped is below 2^-24 of a product, so the error stays that of a 32-bit sum: at most
    sqrt(K) roundings of 2^-24 as they add up at random, with a factor of two; measured 1e-7 to 2e-7."""
    batch, M, N, K = shape
    assert cb.load_library().avhip_gemm_tn_side(4, *shape) == 64
    g = h.rng(31)
    A, B = ((g.standard_normal((batch, K, n)) * scale).astype(np.float32) for n in (M, N))
    got = h.gemm(A, B, np.zeros((batch, M, N), np.float32), "f32", True, False, batched=True)
    want = product(A.astype(np.float64), B.astype(np.float64))
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < max(2 * np.sqrt(K) * 2.0 ** -24, 3e-7)


def test_fp32_values_without_pieces():
    """Infinities, NaN and the largest numbers (no bf16 near them): the sums are those of fp32 products."""
    batch, M, N, K = 130, 64, 64, 300
    assert cb.load_library().avhip_gemm_tn_side(4, batch, M, N, K) == 64
    g = h.rng(32)
    A, B = (g.standard_normal((batch, K, n)).astype(np.float32) for n in (M, N))
    A[3, 7, 5], A[4, 250, 63], B[5, 0, 0], A[6, 20, 20] = np.inf, np.nan, -np.inf, np.finfo(np.float32).max
    B[6, 20] *= 1e-3
    with np.errstate(invalid="ignore", over="ignore"):
        want = product(A.astype(np.float64), B.astype(np.float64))
    got = h.gemm(A, B, np.zeros((batch, M, N), np.float32), "f32", True, False, batched=True)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    rows = np.abs(want).max(axis=2, keepdims=True, where=finite, initial=1.0)
    assert (np.abs(got[finite] - want[finite]) <= 2e-5 * np.broadcast_to(rows, want.shape)[finite]).all()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 2, 2, 1), (16, 32, 32, 16), (16, 34, 62, 15), (9, 30, 98, 257), (3, 64, 66, 129)])
def test_16_bit_pairs_in_small_tiles(oracle, shape, dtype):
    """Every element in its place: values that are whole numbers, so the sums are exact."""
    batch, M, N, K = shape
    g = h.rng(33)
    A, B = (g.integers(-8, 9, (batch, K, n)).astype(np.float64) for n in (M, N))
    got = h.gemm(A, B, np.zeros((batch, M, N)), dtype, True, False, c_dtype="f32", batched=True)
    assert np.array_equal(got, product(A, B))

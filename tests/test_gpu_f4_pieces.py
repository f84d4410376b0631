"""The one-kernel F(4x4, 3x3) in fp32, whose products are of bf16 pieces: no less precise than fp32 products whatever the values are, and the same
answers where values have no pieces.

With nothing in an image but the pixel (3, 3) and in the filters but the tap (0, 0), the transforms leave the values as they are at one point and zeros at
the 35 others, and y(4, 4) is the plain product of the two over the channels."""
import numpy as np
import pytest

import helpers as h
from test_gpu_winograd import ConvShape, f4_forward

pytestmark = pytest.mark.gpu


def product(X, W, alpha=1.0):
    (n, c), k = X.shape, W.shape[0]
    x, w = np.zeros((n, 8, 8, c), np.float32), np.zeros((k, 3, 3, c), np.float32)
    x[:, 3, 3], w[:, 0, 0] = X, W
    return f4_forward(x, w, None, None, ConvShape(n, 8, 8, c, k, 3, 3, 8, 8, -1, -1, 1, 1, 1, 1, 0), alpha1=alpha)[:, 4, 4]


def exact(X, W):
    with np.errstate(invalid="ignore", over="ignore"):
        return X.astype(np.float64) @ W.astype(np.float64).T


def error(got, want):
    return np.linalg.norm(got - want) / np.linalg.norm(want)


@pytest.mark.parametrize("channels", [1, 4, 16, 64])
def test_equal_values(channels):
    """The value whose lower pieces are the largest when they are cut off, not rounded: all that is left out then has one sign.  At most a rounding
    of 2^-24 per channel as they add up at random, and one of the result."""
    v = np.float32(1 + 2.0 ** -7 - 2.0 ** -23)
    X, W = np.full((40, channels), v), np.full((64, channels), v)
    assert error(product(X, W), exact(X, W)) < np.sqrt(channels) * 2.0 ** -24


@pytest.mark.parametrize("x_scale, w_scale", [(0, 0), (-112, 8), (-118, 8), (8, -118), (-124, 20), (-138, 40), (40, -138), (60, 30), (100, -60), (-60, 110)])
def test_values_of_any_size(x_scale, w_scale):
    """Operands down to the subnormal numbers, sums beyond 2^80."""
    g = h.rng(70)
    X, W = ((g.standard_normal((64, 100)) * 2.0 ** e).astype(np.float32) for e in (x_scale, w_scale))
    assert error(product(X, W).astype(np.float64), exact(X, W)) < np.sqrt(100) * 2.0 ** -24


@pytest.mark.parametrize("alpha", [0.0, -2.5, 1.1 * 2.0 ** -89, 1.1 * 2.0 ** -91, 1.1 * 2.0 ** -124, 1.1 * 2.0 ** 100])
def test_factor_of_any_size(alpha):
    """The factor takes the scale of the pieces back, unless it is too small for that."""
    g = h.rng(73)
    X, W = (g.standard_normal((64, 100)).astype(np.float32) for _ in range(2))
    alpha = float(np.float32(alpha))
    want = alpha * exact(X, W)
    assert np.linalg.norm(product(X, W, alpha).astype(np.float64) - want) <= np.sqrt(101) * 2.0 ** -24 * np.linalg.norm(want)


def test_values_without_pieces():
    """In five workgroups; a sum that is no number takes no other with it."""
    g = h.rng(71)
    X, W = g.integers(-3, 4, (40, 37)).astype(np.float32), g.standard_normal((132, 37)).astype(np.float32)
    X[3, 4], X[5, 5], X[6, 6], X[7, 7], X[8, 36] = np.inf, -np.inf, np.nan, np.finfo(np.float32).max, -np.finfo(np.float32).max
    W[:, 7] *= 1e-3
    W[:, 36] *= 1e-38
    W[11, 9] = np.finfo(np.float32).max / 4  # (the weight transform multiplies by up to 4)
    W[12, 12] = 1e-42
    got, want = product(X, W), exact(X, W)
    # beyond the range of a float, and within a rounding of it neither way
    want[np.abs(want) > 3.5e38] = np.inf * np.sign(want[np.abs(want) > 3.5e38])
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    finite = np.isfinite(want)
    size = np.abs(np.nan_to_num(X, nan=0, posinf=0, neginf=0)).astype(np.float64) @ np.abs(W).astype(np.float64).T
    assert (np.abs(got[finite] - want[finite]) <= 37 * 2.0 ** -24 * size[finite]).all()


def test_weights_that_are_no_numbers():
    """The transform makes them infinities of both signs, so that every output of their filters is NaN; the other filters are what they are without them,
    in pieces or, with a filter of such weights in the workgroup, in 32 bits."""
    g = h.rng(72)
    x = g.standard_normal((12, 9, 7, 20)).astype(np.float32)
    w = g.standard_normal((132, 3, 3, 20)).astype(np.float32)
    shape = ConvShape(12, 9, 7, 20, 132, 3, 3, 9, 7, -1, -1, 1, 1, 1, 1, 0)
    want = f4_forward(x, w, None, None, shape)
    w[1, 0, 0, 0], w[2, 1, 1, 2], w[67, 2, 2, 1], w[70, 0, 2, 2] = np.inf, -np.inf, np.inf, np.nan
    got = f4_forward(x, w, None, None, shape)
    odd = np.isin(np.arange(132), (1, 2, 67, 70))
    assert np.isnan(got[..., odd]).all()
    assert error(got[..., ~odd], want[..., ~odd]) < 3e-6
    assert np.array_equal(got[..., 128:], want[..., 128:])

"""ELU of csrc/common.hpp (elu_32), compiled for the host, against 64 bits: at most and on average as far off as the library's function, which is 9e-8 and 1.4e-8 of the value."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from cudabackend_amd import build

SOURCE = """#include "common.hpp"
extern "C" __attribute__((visibility("default"))) void run(const float *x, float *y, int n)
{
	for (int i = 0; i < n; i++)
		y[i] = avhip::elu_32(x[i]);
}
"""


@pytest.fixture(scope="module")
def elu(tmp_path_factory):
    out = tmp_path_factory.mktemp("elu")
    source, target = str(out / "elu.hip"), str(out / "libelu.so")
    with open(source, "w") as f:
        f.write(SOURCE)
    r = subprocess.run(["hipcc", *build.FLAGS, "-I" + build.CSRC, "-shared", source, "-o", target], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-4000:]
    dll = C.CDLL(target)

    def run(x):
        x = np.ascontiguousarray(x, np.float32)
        y = np.empty_like(x)
        dll.run(x.ctypes.data_as(C.c_void_p), y.ctypes.data_as(C.c_void_p), x.size)
        return y
    return run


def test_error(elu):
    bits = np.arange(0x00800000, 0x42D00000, 1021, dtype=np.uint32)  # every 1021st normal float up to 104
    x = -bits.view(np.float32)
    want = np.expm1(x.astype(np.float64))
    error = np.abs(elu(x) / want - 1.0)
    assert error.max() < 9e-8
    for low, high in ((0.001, 0.0625), (0.0625, 0.1), (0.1, 1.0), (1.0, 5.0), (5.0, 104.0)):
        some = (x <= -low) & (x > -high)
        assert error[some].mean() < 2.5e-8  # the rounding of the result alone: up to 2.2e-8, by where the results lie between two powers of 2


def test_special_values(elu):
    x = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 3.5, -1e30, -87.5, 2.0 ** -149, -2.0 ** -149, -2.0 ** -127], np.float32)
    want = np.array([0.0, -0.0, np.inf, -1.0, np.nan, 3.5, -1.0, -1.0, 2.0 ** -149, -2.0 ** -149, -2.0 ** -127], np.float32)
    got = elu(x)
    assert np.array_equal(got, want, equal_nan=True) and np.array_equal(np.signbit(got[:4]), np.signbit(want[:4]))

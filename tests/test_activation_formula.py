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


RUNS = """#include "common.hpp"
template<int ACT, int W> __device__ void run(float *p)
{
	float t[W];
	for (int q = 0; q < W; q++)
		t[q] = p[threadIdx.x * W + q];
	avhip::activate_run<W>(ACT, t);
	for (int q = 0; q < W; q++)
		p[threadIdx.x * W + q] = t[q];
}
extern "C" __global__ void linear_4(float *p) { run<avhip::ACT_LINEAR, 4>(p); }
extern "C" __global__ void linear_16(float *p) { run<avhip::ACT_LINEAR, 16>(p); }
extern "C" __global__ void relu_4(float *p) { run<avhip::ACT_RELU, 4>(p); }
extern "C" __global__ void relu_16(float *p) { run<avhip::ACT_RELU, 16>(p); }
"""


def test_linear_and_relu_are_no_loop(tmp_path):
    """Filters in no whole vectors take LINEAR and RELU through activate_run: LINEAR leaves the values alone, RELU is straight code, however many values a run has."""
    source = str(tmp_path / "runs.hip")
    with open(source, "w") as f:
        f.write(RUNS)
    r = subprocess.run(["hipcc", *build.FLAGS, "-w", "-I" + build.CSRC, "--cuda-device-only", "-S", source, "-o", "-"], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    name, code = None, {}
    for line in r.stdout.splitlines():
        if line.startswith(("linear_", "relu_")) and line.split(":")[0].split("_")[1].isdigit():
            name = line.split(":")[0]
        elif name and line.startswith("\t") and not line.startswith("\t."):
            code.setdefault(name, []).append(line.split()[0])
    assert sorted(code) == ["linear_16", "linear_4", "relu_16", "relu_4"]
    for name, instructions in code.items():
        assert not [i for i in instructions if "cbranch" in i], name
        if name.startswith("linear"):
            assert not [i for i in instructions if i.startswith(("v_max", "v_cmp", "v_cndmask"))], name

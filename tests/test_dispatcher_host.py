"""The dispatcher's way from one plan to the next, on a machine without a GPU: backend.cpp linked with dispatcher_stubs.cpp, in which
"device" memory is host memory and launchers count their calls.  What the plans compute is tested elsewhere."""
import ctypes as C
import os
import subprocess

import pytest

import cudabackend_amd as cb
from cudabackend_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("dispatcher")
    target = str(out / "libdispatcher.so")
    for command in (["hipcc", *build.FLAGS, "-x", "hip", "-c", os.path.join(build.CSRC, "backend.cpp"), "-o", str(out / "backend.o")],
                    ["g++", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-c", os.path.join(HERE, "dispatcher_stubs.cpp"), "-o",
                     str(out / "stubs.o")],
                    ["hipcc", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-Wl,-z,defs", "--offload-arch=" + build.ARCH, "-o", target, str(out / "stubs.o"), str(out / "backend.o")]):
        r = subprocess.run(command, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        assert r.returncode == 0, r.stdout[-4000:]
    dll = C.CDLL(target)
    for name, (res, args) in cb.api.PROTOTYPES.items():
        fn = getattr(dll, name)
        fn.restype, fn.argtypes = res, args
    dll.stub_calls.argtypes = [C.c_char_p]
    dll.stub_set_strided.argtypes = [C.c_int, C.c_double]
    dll.stub_set_direct.argtypes = [C.c_double]
    return dll


class Layer:
    """fp32 3x3 128 -> 128 on 256 images of 15 x 15, in a context of its own: one that the one-kernel F(4x4, 3x3) plan pays for."""

    def __init__(self, lib):
        self.lib = lib
        lib.stub_set(0, 0)
        self.context = self.made(lib.cudaCreateContextDescriptor, 0)
        self.conv = self.made(lib.cudaCreateConvolutionDescriptor)
        cb.check(lib.cudaSetConvolutionDescriptor(self.conv, cb.CONVOLUTION_MODE, 2, (C.c_int * 2)(-1, -1), None, None, 1, None))
        self.x, self.y = self.tensor(256, 15, 15, 128), self.tensor(256, 15, 15, 128)
        self.w = self.tensor(128, 3, 3, 128)
        need = C.c_int64(0)
        cb.check(lib.cudaGetConvolutionWorkspaceSize(self.context, self.conv, self.x[0], self.w[0], 0, C.byref(need)))
        self.space = self.made(lib.cudaCreateMemoryDescriptor, 0, need.value)

    def made(self, create, *args):
        handle = C.c_int64(0)
        cb.check(create(C.byref(handle), *args))
        return handle.value

    def tensor(self, *shape):
        desc, size = self.made(self.lib.cudaCreateTensorDescriptor), 4
        cb.check(self.lib.cudaSetTensorDescriptor(desc, cb.DTYPE_FLOAT32, 4, (C.c_int * 4)(*shape)))
        for n in shape:
            size *= n
        return desc, self.made(self.lib.cudaCreateMemoryDescriptor, 0, size)

    def forward(self, activation=cb.ACTIVATION_RELU, y=None, malloc_fails=False, capturing=False):
        """Status and what was launched."""
        self.lib.stub_set(int(malloc_fails), int(capturing))
        y = y or self.y
        status = self.lib.cudaConvolutionBiasActivationForward(self.context, self.conv, None, self.x[0], self.x[1], self.w[0], self.w[1], 0, 0, None, 0, 0, None,
                                                               y[0], y[1], activation, self.space)
        names = ("f4_weights", "f4", "weights", "input_transform", "gemm", "output_transform", "implicit_gemm")
        return cb.STATUS_NAMES[status], [n for n in names if self.lib.stub_calls(n.encode())]


F4, THREE_PASSES = ["f4"], ["input_transform", "gemm", "output_transform"]


@pytest.fixture()
def layer(lib):
    return Layer(lib)


def test_no_memory_for_the_one_kernel_plans_weights(layer):
    assert layer.forward(cb.ACTIVATION_TANH) == ("SUCCESS", ["weights"] + THREE_PASSES)
    assert layer.forward(malloc_fails=True) == ("SUCCESS", THREE_PASSES), "the plan whose matrices are there takes over"
    assert layer.forward() == ("SUCCESS", ["f4_weights"] + F4)
    assert layer.forward(malloc_fails=True) == ("SUCCESS", F4)


def test_no_memory_for_any_plans_weights(layer):
    assert layer.forward(malloc_fails=True) == ("ALLOC_FAILED", [])
    assert layer.forward() == ("SUCCESS", ["f4_weights"] + F4)


def test_in_place_goes_through_the_workspace(layer):
    """The one-kernel plan writes y while other workgroups still read x."""
    assert layer.forward(y=layer.x) == ("SUCCESS", ["weights"] + THREE_PASSES)


def test_capture_uses_what_is_cached(layer):
    assert layer.forward(capturing=True) == ("SUCCESS", ["implicit_gemm"])
    layer.forward(cb.ACTIVATION_TANH)
    assert layer.forward(capturing=True) == ("SUCCESS", THREE_PASSES)
    layer.forward()
    assert layer.forward(capturing=True) == ("SUCCESS", F4)


class StridedLayer(Layer):
    """bf16 3x3 stride 2, 192 -> 512 on 24 images of 34 x 34: 256 workgroups of the parity-plane kernel, some 29 us by its estimate."""

    def __init__(self, lib):
        self.lib = lib
        lib.stub_set(0, 0)
        self.context = self.made(lib.cudaCreateContextDescriptor, 0)
        self.conv = self.made(lib.cudaCreateConvolutionDescriptor)
        cb.check(lib.cudaSetConvolutionDescriptor(self.conv, cb.CONVOLUTION_MODE, 2, (C.c_int * 2)(-1, -1), (C.c_int * 2)(2, 2), None, 1, None))
        self.x, self.w, self.y = (self.tensor(*shape) for shape in ((24, 34, 34, 192), (512, 3, 3, 192), (24, 17, 17, 512)))
        self.space = 0

    def tensor(self, *shape, offset=0):
        desc, size = self.made(self.lib.cudaCreateTensorDescriptor), 2
        cb.check(self.lib.cudaSetTensorDescriptor(desc, cb.DTYPE_BFLOAT16, 4, (C.c_int * 4)(*shape)))
        for n in shape:
            size *= n
        whole = self.made(self.lib.cudaCreateMemoryDescriptor, 0, size + offset)
        return desc, self.made(self.lib.cudaCreateMemoryView, whole, size, offset) if offset else whole

    def route(self, ring_us, **tensors):
        self.lib.stub_set_strided(256, ring_us)
        for name, t in tensors.items():
            setattr(self, name, t)
        status, _ = self.forward()
        self.lib.stub_set_strided(0, 0.0)
        assert status == "SUCCESS"
        return [n for n in ("strided", "implicit_gemm") if self.lib.stub_calls(n.encode())]


def test_stride_2_layers_go_to_the_ring_kernel_where_that_takes_them(lib):
    """The parity-plane kernel has a layout of its own of the weights, from any address; the ring kernel reads them as they lie, and a layer that
    it declines ends in a kernel that is slower than both."""
    layer = StridedLayer(lib)
    assert layer.route(15.0) == ["implicit_gemm"]
    assert layer.route(40.0) == ["strided"], "slower"
    assert layer.route(0.0) == ["strided"], "declined: switched off, or not far enough below the other kernels"
    assert layer.route(15.0, w=layer.tensor(512, 3, 3, 192, offset=8)) == ["strided"], "weights that are not aligned to 16 bytes"
    layer = StridedLayer(lib)
    images = layer.tensor(24, 34, 34, 192)
    assert layer.route(15.0, x=images, y=(layer.y[0], images[1])) == ["strided"], "in place"


class FusedLayer(Layer):
    """fp32 3x3 32 -> 36 on 34 images of 40 x 43 without a workspace: 306 workgroups of the fused Winograd kernel, 115 us by its estimate."""

    def __init__(self, lib):
        self.lib = lib
        lib.stub_set(0, 0)
        self.context = self.made(lib.cudaCreateContextDescriptor, 0)
        self.conv = self.made(lib.cudaCreateConvolutionDescriptor)
        cb.check(lib.cudaSetConvolutionDescriptor(self.conv, cb.CONVOLUTION_MODE, 2, (C.c_int * 2)(-1, -1), None, None, 1, None))
        self.x, self.w, self.y = (self.tensor(*shape) for shape in ((34, 40, 43, 32), (36, 3, 3, 32), (34, 40, 43, 36)))
        self.space = 0

    def tensor(self, *shape, offset=0):
        desc, memory = super().tensor(*shape)
        if not offset:
            return desc, memory
        size = 4 * shape[0] * shape[1] * shape[2] * shape[3]
        return desc, self.made(self.lib.cudaCreateMemoryView, self.made(self.lib.cudaCreateMemoryDescriptor, 0, size + offset), size, offset)

    def route(self, direct_us, **tensors):
        self.lib.stub_set_direct(direct_us)
        for name, t in tensors.items():
            setattr(self, name, t)
        status, _ = self.forward()
        self.lib.stub_set_direct(0.0)
        assert status == "SUCCESS"
        return [n for n in ("fused", "implicit_gemm") if self.lib.stub_calls(n.encode())]


@pytest.mark.parametrize("direct_us, tensors, want", [
    (50.0, {}, "implicit_gemm"), (150.0, {}, "fused"), (0.0, {}, "fused"),
    (50.0, dict(w=((36, 3, 3, 32), 4)), "fused"), (50.0, dict(w=((36, 3, 3, 32), 16)), "implicit_gemm"), (50.0, dict(x=((34, 40, 43, 32), 8)), "fused"),
    (50.0, dict(y=((34, 40, 43, 36), 4)), "implicit_gemm"), (50.0, dict(x=((34, 40, 43, 36), 0), w=((36, 3, 3, 36), 0), y="x"), "fused")], ids=str)
def test_direct_sums_replace_the_fused_kernel_where_they_read_the_operands(lib, direct_us, tensors, want):
    """The fused kernel has a layout of its own of the weights, from any address; the direct kernels read them as they lie, and what they decline ends in a kernel that is slower than
    both.  Nor do calls in place go to them, nor any where they are not weighed."""
    layer = FusedLayer(lib)
    made = {name: layer.tensor(*t[0], offset=t[1]) for name, t in tensors.items() if t != "x"}
    if tensors.get("y") == "x":
        made["y"] = made["x"]
    assert layer.route(direct_us, **made) == [want]

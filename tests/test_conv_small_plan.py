"""What the kernel of small tiles (csrc/conv_small.hip, csrc/conv_small16.hip) is estimated to take, and what it gets by that.  Host arithmetic only."""
import ctypes as C

import pytest

import cudabackend_amd as cb


class Shape(C.Structure):
    _fields_ = [(n, C.c_int) for n in "N H W C K R S Ho Wo pad_h pad_w stride_h stride_w dil_h dil_w mode".split()]


VECTORS, ELEMENTS, ACTIVATION = range(3)  # how results leave: HandOver of csrc/conv_small.hpp
CODE = {"f32": cb.DTYPE_FLOAT32, "f16": cb.DTYPE_FLOAT16, "bf16": cb.DTYPE_BFLOAT16, "i8": cb.DTYPE_INT8}


def shape_of(n, h, w, c, k, r, stride):
    return Shape(n, h, w, c, k, r, r, *((v + 2 * (r // 2) - r) // stride + 1 for v in (h, w)), -(r // 2), -(r // 2), stride, stride, 1, 1, 0)


@pytest.fixture()
def lib():
    dll = cb.load_library()
    dll.avhip_conv2d_small_us.restype = C.c_double
    dll.avhip_set_small_problem_threshold.restype = C.c_int
    previous = dll.avhip_set_small_problem_threshold(4096)
    yield dll
    dll.avhip_set_small_problem_threshold(previous)


def us(lib, layer, hand_over, dtype="f32"):
    return lib.avhip_conv2d_small_us(CODE[dtype], C.byref(shape_of(*layer)), hand_over)


def test_the_estimate_is_of_the_kernel_that_the_call_reaches(lib):
    """What the dispatcher weighs the fused Winograd kernel against in fp32: single filters and activations cost more than whole vectors, fp32 with both, in the general gather kernel, the most."""
    small, large = (34, 40, 43, 32, 36, 3, 1), (168, 31, 31, 256, 512, 3, 1)
    assert 0.0 < us(lib, small, VECTORS) < us(lib, small, ELEMENTS) <= us(lib, small, ACTIVATION)
    assert 0.0 < us(lib, large, VECTORS) < us(lib, large, ELEMENTS) < us(lib, large[:4] + (509, 3, 1), ACTIVATION)
    assert us(lib, small[:3] + (34, 36, 3, 1), VECTORS) == 0.0  # channels in no whole chunks
    for switch in (0, -1):
        lib.avhip_set_small_problem_threshold(switch)
        assert us(lib, small, VECTORS) == us(lib, large, VECTORS) == 0.0

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


# dtype; images, rows, columns, channels, filters, their size, stride; microseconds without and in tiles of 16 x 16: one to four of them to a compute unit and more, short and long k, rows that are
# whole lines of 128 bytes and not, layers that were split, one tap, few channels
TIMED = [("f16", (1, 15, 15, 128, 128, 3, 1), 5.9, 4.1), ("f32", (8, 15, 15, 64, 64, 3, 1), 8.3, 5.7), ("f32", (2, 16, 16, 128, 128, 3, 1), 11.1, 5.7),
         ("i8", (1, 16, 20, 48, 48, 1, 1), 3.6, 2.7), ("f16", (3, 13, 13, 256, 256, 3, 1), 7.9, 6.6), ("f16", (2, 18, 18, 384, 128, 5, 1), 19.5, 14.7), ("bf16", (3, 20, 20, 128, 128, 3, 1), 6.5, 5.7),
         ("bf16", (6, 10, 9, 256, 120, 5, 1), 13.2, 11.3), ("f16", (1, 29, 28, 304, 352, 3, 1), 12.9, 15.6), ("f16", (75, 19, 22, 296, 32, 3, 2), 12.7, 14.4), ("f16", (34, 10, 13, 104, 64, 5, 1), 12.0, 13.5),
         ("bf16", (16, 19, 18, 472, 192, 3, 2), 18.3, 24.4), ("bf16", (4, 45, 46, 224, 32, 5, 1), 19.5, 24.8), ("f16", (7, 27, 26, 384, 200, 5, 2), 23.7, 36.2), ("bf16", (78, 9, 12, 416, 32, 3, 1), 14.9, 17.0),
         ("f16", (72, 38, 38, 256, 16, 3, 1), 51.8, 57.7), ("f16", (2, 51, 51, 160, 192, 3, 2), 7.5, 8.6), ("f16", (14, 14, 14, 96, 96, 3, 1), 5.6, 6.4), ("i8", (19, 16, 12, 80, 64, 3, 1), 4.5, 4.9),
         ("bf16", (42, 22, 18, 64, 64, 1, 1), 4.2, 4.6), ("i8", (35, 18, 20, 128, 80, 1, 1), 4.1, 4.6), ("i8", (20, 18, 20, 80, 80, 1, 1), 4.3, 4.0), ("i8", (19, 11, 16, 192, 192, 1, 1), 4.8, 4.1),
         ("f16", (98, 8, 7, 24, 48, 5, 1), 16.6, 5.5), ("f16", (8, 22, 27, 4, 128, 5, 2), 7.1, 4.0), ("f32", (6, 11, 11, 4, 192, 3, 1), 9.1, 3.4), ("bf16", (2, 45, 50, 2, 96, 5, 1), 6.6, 5.4)]


@pytest.mark.parametrize("dtype, layer, without, within", TIMED)
def test_tiles_of_16_x_16_where_they_are_faster(lib, dtype, layer, without, within):
    plan = lib.avhip_conv2d_plain_small_plan(CODE[dtype], C.byref(shape_of(*layer)))
    assert (plan in (9, 12, 16)) == (within < without), plan


@pytest.mark.parametrize("dtype, layer", [("bf16", (32, 224, 224, 3, 64, 7, 2)), ("f32", (10, 137, 137, 3, 96, 5, 1)), ("f16", (256, 15, 15, 4, 128, 3, 1)), ("f16", (94, 25, 25, 16, 128, 3, 1)),
                                          ("i8", (60, 28, 28, 16, 64, 3, 1)), ("f32", (64, 56, 56, 8, 64, 3, 1))])
def test_few_channels_of_many_pixels_stay_in_the_kernels_made_for_them(lib, dtype, layer):
    assert lib.avhip_conv2d_plain_small_plan(CODE[dtype], C.byref(shape_of(*layer))) == 0

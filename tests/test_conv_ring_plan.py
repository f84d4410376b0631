"""Which 16-bit layers of few filters the kernel with a ring of LDS buffers (csrc/conv_ring.hip) takes from the small tiles: layers timed with both go to the
faster one.  Host arithmetic only."""
import ctypes as C

import pytest

import cudabackend_amd as cb


class Shape(C.Structure):
    _fields_ = [(n, C.c_int) for n in "N H W C K R S Ho Wo pad_h pad_w stride_h stride_w dil_h dil_w mode".split()]


VECTORS, ELEMENTS, ACTIVATION = range(3)  # how results leave: HandOver of csrc/conv_small.hpp

# n, h, w, c, k, r, stride, hand-over, residual; microseconds without the ring kernel and in it
TIMED = [((65, 15, 15, 320, 14, 5, 1, ELEMENTS, True), 22.9, 32.5), ((187, 10, 11, 512, 13, 1, 1, ELEMENTS, True), 7.7, 10.2),
         ((94, 30, 30, 400, 10, 3, 1, ELEMENTS, True), 58.2, 70.5), ((160, 21, 22, 320, 14, 3, 1, ELEMENTS, False), 39.6, 46.6),
         ((99, 37, 33, 192, 12, 3, 2, ACTIVATION, False), 15.4, 17.9), ((204, 24, 20, 80, 12, 3, 1, ACTIVATION, False), 17.7, 20.3),
         ((202, 44, 47, 88, 18, 3, 1, ACTIVATION, True), 78.6, 90.1), ((33, 62, 63, 368, 12, 1, 1, ACTIVATION, False), 21.7, 24.2),
         ((63, 33, 36, 224, 14, 3, 1, ELEMENTS, True), 33.9, 37.5), ((136, 51, 52, 72, 10, 3, 1, ACTIVATION, False), 52.6, 57.8),
         ((158, 27, 23, 64, 16, 3, 1, ACTIVATION, False), 15.7, 17.2), ((95, 32, 35, 320, 20, 3, 1, ACTIVATION, False), 56.4, 61.7),
         ((16, 40, 40, 64, 20, 5, 1, VECTORS, True), 13.3, 10.8), ((15, 42, 45, 64, 16, 5, 1, VECTORS, False), 17.7, 10.2),
         ((223, 58, 58, 64, 12, 3, 1, VECTORS, True), 237.1, 80.5), ((236, 51, 51, 32, 12, 3, 1, ACTIVATION, True), 281.1, 81.1),
         ((79, 26, 26, 224, 112, 3, 1, ACTIVATION, False), 54.4, 43.5), ((37, 19, 17, 72, 100, 3, 1, ACTIVATION, True), 12.0, 10.0)]


@pytest.mark.parametrize("layer, without, within", TIMED)
def test_the_faster_kernel_is_taken(layer, without, within):
    n, h, w, c, k, r, stride, hand_over, residual = layer
    shape = Shape(n, h, w, c, k, r, r, *((v + 2 * (r // 2) - r) // stride + 1 for v in (h, w)), -(r // 2), -(r // 2), stride, stride, 1, 1, 0)
    plan = cb.load_library().avhip_conv2d_ring_plan(cb.DTYPE_FLOAT16, cb.DTYPE_FLOAT16, C.byref(shape), hand_over, int(residual))
    assert (plan >= 0) == (within < without)

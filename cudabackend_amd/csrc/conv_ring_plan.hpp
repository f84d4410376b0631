/*
 * conv_ring_plan.hpp -- what the dispatcher and tests may ask of the kernel with a ring of LDS buffers (conv_ring.hip).
 */
#ifndef AVHIP_CONV_RING_PLAN_HPP_
#define AVHIP_CONV_RING_PLAN_HPP_

#include "../../include/avocado_hip_kernels.h"

extern "C"
{
	/* The microseconds the kernel is estimated to take for a call of avhip_conv2d_implicit_gemm, or 0 where that goes to another kernel, given 16-byte
	 * aligned x and w below 2 GiB, a zero padding value and y apart from x.  `hand_over`: 0 LINEAR or RELU in whole aligned vectors of four
	 * filters, 1 those element by element, 2 any other activation; `residual`: whether there is a z. */
	AVHIP_API double avhip_conv2d_ring_us(int x_dtype, int y_dtype, const avhipConvShape *shape, int hand_over, int residual);
	/* The tile that such a call gets, pixels x filters: 0 256 x 128, 1 128 x 128, 2 128 x 64, 3 64 x 64, or -1 where it goes to another kernel. */
	AVHIP_API int avhip_conv2d_ring_plan(int x_dtype, int y_dtype, const avhipConvShape *shape, int hand_over, int residual);
}

#endif /* AVHIP_CONV_RING_PLAN_HPP_ */

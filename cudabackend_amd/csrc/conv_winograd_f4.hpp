/*
 * conv_winograd_f4.hpp -- internal interface of the one-kernel Winograd F(4x4, 3x3) in fp32 (conv_winograd_f4.hip).  The functions are
 * exported so that a test can call them with layers the dispatcher would send elsewhere.
 */
#ifndef AVHIP_CONV_WINOGRAD_F4_HPP_
#define AVHIP_CONV_WINOGRAD_F4_HPP_

#include "../../include/avocado_hip_kernels.h"

extern "C"
{
	/* y = act(alpha1 * conv(x, w) + bias + alpha2 * z) in fp32: 3x3, stride 1, dilation 1, output of the input's size, zero padding value, any
	 * number of channels, K a multiple of four, y and z aligned to 16 bytes, x below 512 MiB, U below 768 MiB and y below 2 GiB, beta = 0, LINEAR or RELU,
	 * y apart from x; AVHIP_NOT_SUPPORTED for other layers, with nothing launched.  Stands where the reference calls its non-fused
	 * kernels one after another, src/winograd_nonfused.cu:609-877.  U is what avhip_winograd_f4_weight_transform wrote (taps reversed when
	 * `invert`): avhip_winograd_f4_weight_bytes(K, C) bytes, [K / 32][36][C / 16][3 pieces][64 lanes][8] bf16, the pieces adding up to 2^16 times the
	 * value or, where it is no number or too large, a NaN and the value's own bits; K and C filled up to multiples of 64 and 16 with zeros. */
	AVHIP_API int avhip_conv2d_winograd_f4(void *stream, const avhipConvShape *shape, const void *x, const void *U, const void *bias, const void *z, void *y,
			double alpha1, double alpha2, double beta, int activation);
	AVHIP_API int avhip_winograd_f4_weight_transform(void *stream, int invert, const void *w, void *U, int K, int C);
	AVHIP_API int64_t avhip_winograd_f4_weight_bytes(int K, int C);
}

namespace avhip
{
	/* Whether avhip_conv2d_winograd_f4 takes the layer (U aligned to 16 bytes, y apart from x): to be asked before the weights are transformed. */
	bool winograd_f4_takes(const avhipConvShape &s, const void *x, const void *z, const void *y, double beta, int activation);
}

#endif /* AVHIP_CONV_WINOGRAD_F4_HPP_ */

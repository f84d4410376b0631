/*
 * conv_small.hpp -- internal interface of the small-problem implicit-GEMM kernel (conv_small.hip).
 */
#ifndef AVHIP_CONV_SMALL_HPP_
#define AVHIP_CONV_SMALL_HPP_

#include "conv_epilogue.hpp"

namespace avhip
{
	/* Launches the kernel and returns true when its estimate for the problem is below that of the kernels with 128 x 128 (or
	 * 256 x 64) workgroup tiles; returns false without side effects otherwise.  The caller has established the conditions of the
	 * branch-free loaders (16-byte aligned tensors below 2 GiB, zero padding value);
	 * any activation and number of filters. */
	template<typename TE, typename Epi>
	bool conv_small_launch(hipStream_t stream, const avhipConvShape &s, const void *x, const void *w, const Epi &epi);

	/* tiles x tiles MFMA tiles of 32 x 32, `waves` wavefronts sharing the k range, and the estimated microseconds */
	struct SmallPlan
	{
		int tiles, waves;
		double us;
	};
	int conv_small_threshold(); /* what avhip_set_small_problem_threshold set */
	SmallPlan conv_small_plan(const avhipConvShape &s, int element_bytes);
	/* Whether the launcher sends the layer to that kernel, given the conditions above.  `plain`: LINEAR or RELU, whole aligned
	 * vectors of four filters. */
	bool conv_small_preferred(const avhipConvShape &s, int element_bytes, bool plain);
}

#endif /* AVHIP_CONV_SMALL_HPP_ */

/*
 * conv_ring.hpp -- internal interface of the implicit-GEMM kernel with a ring of LDS buffers (conv_ring.hip).
 */
#ifndef AVHIP_CONV_RING_HPP_
#define AVHIP_CONV_RING_HPP_

#include "conv_small.hpp"

namespace avhip
{
	/* The microseconds the kernel is estimated to take, or 0 where the layer is left to the others: those are no slower by their estimates, or
	 * it is one that the kernel cannot run (16-bit and 8-bit types, channels of whole 16-byte chunks).  `small`: conv_small_choice of the call. */
	double conv_ring_us(const avhipConvShape &s, int element_bytes, int out_bytes, const SmallChoice &small, bool residual);

	/* Launches the kernel and returns true where conv_ring_us is not 0; returns false without side effects otherwise.  The caller has established
	 * the conditions of the branch-free loaders (16-byte aligned tensors below 2 GiB, zero padding value); any activation and number of
	 * filters.  Calls that work in place are left to the other kernels. */
	template<typename TE, typename Epi>
	bool conv_ring_launch(hipStream_t stream, const avhipConvShape &s, const void *x, const void *w, const Epi &epi, const SmallChoice &small);
}

#endif /* AVHIP_CONV_RING_HPP_ */

/*
 * conv_ring_plan.hpp -- which tile the kernel with a ring of LDS buffers (conv_ring.hip) takes for a layer, and how long that is estimated to
 * take: host arithmetic only, for its launcher and for the dispatcher.
 */
#ifndef AVHIP_CONV_RING_PLAN_HPP_
#define AVHIP_CONV_RING_PLAN_HPP_

#include <cmath>

#include "../../include/avocado_hip_kernels.h"

namespace avhip
{
	struct RingPlan
	{
		int pixels, filters, per_cu; /* of a tile; workgroups that share a compute unit */
		/* microseconds: of a launch, of a stage per workgroup on the compute unit, of a workgroup's beginning and end, more for results element by
		 * element and for those with a call per activation, and per megabyte of results and residuals */
		double launch, stage, tile, elements, activation, megabyte;
	};
	/* Fitted to 410 layers of 16-bit and 8-bit types (36 to 500000 pixels, 16 to 1024 channels and filters, 1x1 to 5x5, strides 1 and 2), each timed with
	 * every plan; root mean square error 9 to 12 %.  The four are needed: the best plan is each of them on a fifth of the layers at least, without
	 * the second the mean gain falls from 12 to 11 %, without the first from 12 to 10. */
	constexpr RingPlan RING_PLANS[] = { { 256, 128, 1, 0.0, 0.63, 5.5, 7.4, 10.0, 0.07 }, { 128, 128, 1, 1.1, 0.38, 3.5, 3.8, 4.6, 0.045 },
			{ 128, 64, 2, 2.1, 0.265, 2.0, 1.8, 2.8, 0.04 }, { 64, 64, 3, 2.5, 0.165, 1.7, 1.7, 2.6, 0.0 } };

	struct RingChoice
	{
		int plan;
		double us;
	};
	/* `hand_over`: 0 whole vectors, 1 element by element, 2 any activation (HandOver of conv_small.hpp) */
	inline RingChoice ring_choice(const avhipConvShape &s, int element_bytes, int out_bytes, int hand_over, bool residual)
	{
		const double pixels = static_cast<double>(s.N) * s.Ho * s.Wo;
		const double stages = std::ceil(static_cast<double>(s.R) * s.S * (s.C * element_bytes / 16) / 8.0);
		const double megabytes = pixels * s.K * out_bytes * (residual ? 2.0e-6 : 1.0e-6);
		RingChoice best = { -1, 0.0 };
		for (int i = 0; i < 4; i++)
		{
			const RingPlan &p = RING_PLANS[i];
			const double tile = p.tile + (hand_over == 1 ? p.elements : hand_over == 2 ? p.activation : 0.0);
			const double loads = std::ceil(pixels / p.pixels) * ((s.K + p.filters - 1) / p.filters) / 256.0; /* of workgroups, one per compute unit each */
			const double rounds = std::floor(loads / p.per_cu), rest = std::ceil(loads - rounds * p.per_cu);
			const double us = p.launch + (rounds + (rest > 0.0 ? 1.0 : 0.0)) * tile + (rounds * p.per_cu + rest) * p.stage * stages + p.megabyte * megabytes;
			if (best.plan < 0 || us < best.us)
				best = { i, us };
		}
		return best;
	}
}

#endif /* AVHIP_CONV_RING_PLAN_HPP_ */

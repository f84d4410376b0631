/*
 * conv_small.hpp -- internal interface of the small-problem implicit-GEMM kernel (conv_small.hip).
 */
#ifndef AVHIP_CONV_SMALL_HPP_
#define AVHIP_CONV_SMALL_HPP_

#include "conv_epilogue.hpp"
#include "conv_estimates.hpp"
#include "conv_pointwise.hpp"

namespace avhip
{
	struct SmallGeom
	{
		int H, W, C, K, R, S, Ho, Wo, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, flip;
		int chunks_per_tap; /* 16-byte chunks of the channels of one tap */
		unsigned int by_chunks, by_s; /* ceil(2^32 / chunks_per_tap), ceil(2^16 / S): division by multiplication */
		int pixels, images;
		unsigned int pixel_tiles, filter_tiles;
		Divisor by_wo, by_ho, by_tiles; /* by_tiles: of the faster of the two */
		int pixels_first; /* order of the tiles: pixel tiles run fastest within an XCD (more weights than image), or filter tiles */
	};
	/* The geometry of a launch of so many tiles, below 2^31 of them and of pixels. */
	inline SmallGeom small_geometry(const avhipConvShape &s, int element_bytes, int64_t pixel_tiles, int64_t filter_tiles)
	{
		const int64_t pixels = static_cast<int64_t>(s.N) * s.Ho * s.Wo;
		SmallGeom g;
		g.H = s.H;
		g.W = s.W;
		g.C = s.C;
		g.K = s.K;
		g.R = s.R;
		g.S = s.S;
		g.Ho = s.Ho;
		g.Wo = s.Wo;
		g.pad_h = s.pad_h;
		g.pad_w = s.pad_w;
		g.stride_h = s.stride_h;
		g.stride_w = s.stride_w;
		g.dil_h = s.dil_h;
		g.dil_w = s.dil_w;
		g.flip = s.mode != 0 ? 1 : 0;
		g.chunks_per_tap = (s.C * element_bytes + 15) / 16;
		g.by_chunks = static_cast<unsigned int>(((1ll << 32) + g.chunks_per_tap - 1) / g.chunks_per_tap); /* 1: unused */
		g.by_s = (65536 + s.S - 1) / s.S;
		g.pixels = static_cast<int>(pixels);
		g.images = s.N;
		g.pixels_first = static_cast<int64_t>(s.K) * s.R * s.S > static_cast<int64_t>(s.N) * s.H * s.W ? 1 : 0;
		g.pixel_tiles = static_cast<unsigned int>(pixel_tiles);
		g.filter_tiles = static_cast<unsigned int>(filter_tiles);
		g.by_wo = divisor(s.Wo);
		g.by_ho = divisor(s.Ho);
		g.by_tiles = divisor(g.pixels_first ? g.pixel_tiles : g.filter_tiles);
		return g;
	}

	/* Whether the call writes y where x lies.  No header promises that, but it works where the sums are complete before the first result
	 * is written (k split through the workspace, the three passes of non-fused Winograd) and where a workgroup alone reads the pixels that
	 * it writes (one-tap filters, up to 128 filters in the kernels with 128 x 128 tiles).  Neither holds for tiles of 32 x 32 or 64 x 64. */
	inline bool in_place(const avhipConvShape &s, const void *x, int x_size, const void *y, int y_size)
	{
		const int64_t x_bytes = static_cast<int64_t>(s.N) * s.H * s.W * s.C * x_size, y_bytes = static_cast<int64_t>(s.N) * s.Ho * s.Wo * s.K * y_size;
		const char *in = static_cast<const char*>(x), *out = static_cast<const char*>(y);
		return in < out + y_bytes && out < in + x_bytes;
	}

	/* Layers of few input channels, below 64 bytes per pixel, whose (tap, channel) pairs are worth packing into the k-steps instead of spending a step
	 * per tap, given whole aligned vectors of results and LINEAR or RELU.  At 64 (half a k-step per tap) the other kernels are the faster ones, measured on
	 * 3x3 layers of 64 int8 / 32 bf16 / 16 fp32 channels (12 against 28 us, 21 against 52 us, 82 against 113 us); at 48 and 32 bytes those
	 * that pack are (16 against 22 us, 13 against 22 us). */
	inline bool conv_few_channels(const avhipConvShape &s, int element_bytes)
	{
		return static_cast<int64_t>(s.C) * element_bytes < 64 && s.R * s.S > 1;
	}

	int conv_small_threshold(); /* what avhip_set_small_problem_threshold set */
	bool conv_small_possible(const avhipConvShape &s, int element_bytes); /* taps and chunks of a tap within the kernel's arithmetic */
	/* How results leave: LINEAR or RELU in whole aligned vectors of four filters; those activations element by element; any activation */
	enum class HandOver
	{
		PLAIN, ELEMENTS, ACTIVATION
	};
	/* What the launchers of this kernel and of the ring kernel (conv_ring.hip) both ask about a call, worked out once: the host bounds the smallest layers, at
	 * some 5 us a call, of which the choice of a kernel took 148 ns with each of the two on its own, 60 so. */
	struct SmallChoice
	{
		HandOver hand_over;
		double one_tap_us; /* conv_pointwise_us */
		bool preferred; /* whether the layer is sent to this kernel: its estimate is below that of the kernels with 128 x 128 (or 256 x 64) workgroup tiles */
		SmallPlan plan;
		double us; /* estimate of the layer in this kernel or, where it is not preferred, in those (0: it cannot run the layer) */
		bool larger_preferred; /* the same two without tiles of 16 x 16 */
		double larger_us;
	};
	SmallChoice conv_small_choice(const avhipConvShape &s, int element_bytes, HandOver hand_over, double one_tap_us);
	template<typename TE, typename Epi>
	SmallChoice conv_small_choice(const avhipConvShape &s, const Epi &epi)
	{
		/* whole 4-filter vectors and LINEAR / RELU, or anything (the integer epilogues know no other activation) */
		const bool simple = is_simple_activation(epi.activation);
		const HandOver hand_over = !simple ? HandOver::ACTIVATION : epi.vec ? HandOver::PLAIN : HandOver::ELEMENTS;
		return conv_small_choice(s, static_cast<int>(sizeof(TE)), hand_over, hand_over == HandOver::PLAIN ? conv_pointwise_us<TE>(s, epi) : 0.0);
	}
	/* The kernel of 16 x 16 tiles (conv_small16.hip), for conv_small_launch. */
	template<typename TE, typename Epi>
	void conv_small16_launch(hipStream_t stream, const dim3 &grid, int waves, const void *x, const void *w, const SmallGeom &g, const Epi &epi, HandOver hand_over);
	/* Launches the kernel and returns true where it is preferred; returns false without side effects otherwise.  The caller has established the conditions of
	 * the branch-free loaders (16-byte aligned tensors below 2 GiB, zero padding value); any activation and number of filters.  Calls
	 * that work in place are left to the other kernels. */
	template<typename TE, typename Epi>
	bool conv_small_launch(hipStream_t stream, const avhipConvShape &s, const void *x, const void *w, const Epi &epi, const SmallChoice &choice);
	/* fp32 layers that the image-tile kernel takes: whether the gather kernel, whose fp32 products are of bf16 pieces, is estimated to be faster. */
	bool conv_gather_before_image_tiles(const avhipConvShape &s);
}

#endif /* AVHIP_CONV_SMALL_HPP_ */

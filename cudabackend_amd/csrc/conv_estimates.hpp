/*
 * conv_estimates.hpp -- what the implicit-GEMM kernels of small tiles (conv_small.hip) and of 128 x 128 tiles are estimated to take: host arithmetic on a shape, for their
 * launchers and for the dispatcher, which weighs other plans against them.
 */
#ifndef AVHIP_CONV_ESTIMATES_HPP_
#define AVHIP_CONV_ESTIMATES_HPP_

#include <algorithm>
#include <cmath>
#include <stdint.h>

#include "../../include/avocado_hip_kernels.h"

extern "C"
{
	/* Microseconds that a layer of more than one tap in 16-byte chunks of channels is estimated to take in the implicit-GEMM kernel that it is sent to, small tiles or 128 x 128 (256 x 64) ones; 0 where
	 * neither is weighed (avhip_set_small_problem_threshold at 0 or below).  `hand_over`: HandOver of conv_small.hpp.  Defined in conv_small.hip. */
	AVHIP_API double avhip_conv2d_small_us(int x_dtype, const avhipConvShape *shape, int hand_over);
}

namespace avhip
{
	/* tiles of side x side, `waves` wavefronts sharing the k range, and the estimated microseconds */
	struct SmallPlan
	{
		int side, waves;
		double us;
		double larger_us; /* of the best without tiles of 16 x 16; 0: there is none */
		int waves_16; /* and of the best with them */
		double us_16;
		SmallPlan of_16() const
		{
			return { 16, waves_16, us_16, larger_us, waves_16, us_16 };
		}
	};
	struct SmallTiling
	{
		int side_bits, wave_bits; /* a side of 2^side_bits: shifts on the host, not divisions or calls that round */
	};
	inline constexpr SmallTiling PLANS[] = { { 5, 0 }, { 5, 2 }, { 5, 3 }, { 6, 2 }, { 4, 0 }, { 4, 2 }, { 4, 3 } };

	struct Pace
	{
		double launch, chain, stage, tile;
	};
	/* Microseconds: launch and first loads, one stage of a wavefront alone, one stage of a tile when its compute unit is busy, and everything
	 * else about a tile.  Order of PLANS.  16-bit and 8-bit types: the larger of the two stage costs, fitted to 320 layers (7 to 64 rows and
	 * columns, 16 to 512 channels and filters, 1x1 to 5x5, up to 12 GFLOP; root mean square error 6 to 14 %).  fp32: the root of the sum of
	 * their squares, fitted to 222 layers timed with every plan (up to 6 GFLOP): the plan chosen is 0.5 % slower than the best of the four
	 * on average and 15 % at most, with the larger of the two 1.2 % and 36 % (52 -> 408 1x1 on 637 pixels: 7.2 us with four wavefronts, which that chose,
	 * 5.5 with one).  The tiles of 64 x 64, whose products are of bf16 pieces, to 260 layers (6 %), and
	 * 6 % and 0.6 us more than that: then none of the 43 that get them is slower than with what it got before (1.28 times as fast on average; without
	 * that 56, four of them slower).  The tiles of 16 x 16 (conv_small16.hip; the root of the sum of squares in every type) to 254 layers of up to 800 tiles of 32 x 32, 6 to 8 %, and taken
	 * where they are 5 % below the others; in 16 and 8 bits by margin_16. */
	inline constexpr Pace PACE_16[] = { { 4.99, 0.303, 0.107, 0.20 }, { 3.34, 0.409, 0.084, 0.90 }, { 2.64, 0.173, 0.091, 2.40 }, { 3.41, 0.88, 0.182, 1.86 },
			{ 2.75, 0.171, 0.043, 0.09 }, { 2.81, 0.144, 0.041, 0.205 }, { 2.31, 0.228, 0.035, 0.73 } };
	inline constexpr Pace PACE_32[] = { { 3.80, 0.647, 0.143, 0.37 }, { 3.19, 0.490, 0.149, 1.00 }, { 2.34, 0.162, 0.165, 2.98 }, { 4.34, 1.13, 0.371, 3.14 },
			{ 2.91, 0.280, 0.069, 0.05 }, { 2.83, 0.217, 0.060, 0.275 }, { 2.65, 0.260, 0.058, 0.52 } };

	/* How far below those of larger tiles the estimate of tiles of 16 x 16 has to be: 5 %, and in 16 and 8 bits, whose larger tiles are estimated 5 to 10 % too high where their number begins a second round or k is long, 10 beyond
	 * four to a compute unit (three, or a long k, in rows that are no whole lines), 20 for many tiles of a long k.  Of 1794 16-bit layers that got tiles of 16 x 16 with 5 % everywhere, a tile beyond four in part and no look at
	 * how rows lie, 74 were more than 3 % slower with them, by 25 at most (472 -> 192 3x3 stride 2 on 16 x 19 x 18 18.3 -> 24.4 us; 384 -> 200 5x5 stride 2 on 7 x 27 x 26, which was split before, 23.7 -> 36.2).
	 * 1584 keep them, 10 of those more than 3 % slower, by 10 at most, and 1.26 times as fast on average. */
	inline double margin_16(int element_bytes, bool whole_lines, int64_t tiles, int64_t stages)
	{
		if (element_bytes == 4 || tiles <= 256 || (whole_lines ? tiles <= 1024 : tiles <= 768 && stages < 90))
			return 0.95;
		return tiles <= 1536 || stages < 24 ? 0.9 : 0.8;
	}

	/* The kernels with 128 x 128 (image-tile kernel: 256 x 64) workgroup tiles: launch, a round of 512 workgroups (two to a compute unit), and
	 * a k-step of one that has a compute unit to itself or shares it.  The last round, if it is of up to 256, goes at the pace of the former.
	 * Microseconds, fitted to 448 layers (2000 to 130000 pixels, 16 to 512 channels and filters; root mean square error 6 to 13 %).  With every
	 * round of the same length a 517th workgroup seemed to double the time: fp16 128 -> 128 3x3 on 129 images of 18 x 18 went to small tiles
	 * and took 29.3 us, 25.5 in the image-tile kernel.  The image tiles' figures hold where filters fill blocks of 64 and channels 128 bytes; of 18 layers
	 * where they do not, seven take 1.3 to 1.9 times as long (fp16 224 -> 112 3x3 on 79 x 26 x 26 28.5 : 49 us), and int8
	 * layers up to a third longer (128 -> 128 on 128 x 20 x 20 10.1 : 13). */
	struct TilePace
	{
		double launch, round, alone, shared;
	};
	enum TileKernel
	{
		IMAGE_TILES, GATHER, GATHER_BY_ELEMENTS, GATHER_ACTIVATION, GATHER_GENERAL
	};
	inline constexpr TilePace TILES_16[] = { { 0.0, 4.0, 0.42, 0.68 }, { 1.7, 7.7, 0.70, 0.90 }, { 0.0, 13.5, 0.69, 0.96 }, { 4.4, 15.9, 0.67, 0.88 } };
	/* (fp32 in the gather kernel: products of bf16 pieces, 144 layers without a residual, 5 % with rounds of 9.2 us; not in its general instance, which takes an activation and filters in no whole
	 * vectors at once) */
	inline constexpr TilePace TILES_32[] = { { 3.0, 4.1, 1.94, 3.84 }, { 2.5, 11.5, 1.67, 2.50 }, { 0.3, 17.3, 1.67, 2.50 }, { 4.7, 18.0, 1.67, 2.50 }, { 4.7, 18.0, 2.07, 3.92 } };

	/* Tiles of an image in the image-tile kernel, whose tiles are rectangles and lie at the pitch of their halo: 53 columns make tiles of 4 rows, 14 of them and not the 11 that hold
	 * as many pixels.  With those 11, 64 -> 256 3x3 on 5 x 53 x 53 in fp32 seemed to fit one workgroup to a compute unit, 42 us, and took 77 (57.9 in the fused Winograd kernel). */
	inline int image_tiles(const avhipConvShape &s)
	{
		int best = 0;
		for (int parts = 1; parts <= 4; parts++)
		{
			const int columns = (s.Wo + parts - 1) / parts, pitch = columns + s.S - 1;
			if (columns > 256)
				continue;
			const int rows = std::min(s.Ho, 1 + (256 - columns) / pitch), tiles = parts * ((s.Ho + rows - 1) / rows);
			best = best == 0 || tiles < best ? tiles : best;
		}
		return best != 0 ? best : (s.Ho * s.Wo + 255) / 256;
	}
	inline double tile_kernel_us(const avhipConvShape &s, int element_bytes, int kernel)
	{
		const double pixels = static_cast<double>(s.N) * s.Ho * s.Wo;
		const double steps = static_cast<double>(s.R) * s.S * ((s.C * element_bytes + 127) / 128);
		const TilePace &pace = (element_bytes == 4 ? TILES_32 : TILES_16)[kernel];
		double workgroups = std::ceil(pixels / 128.0) * ((s.K + 127) / 128);
		if (kernel == IMAGE_TILES)
			workgroups = static_cast<double>(s.N) * ((s.K + 63) / 64) * (element_bytes == 4 ? image_tiles(s) : (s.Ho * s.Wo + 255) / 256);
		const double rounds = std::floor(workgroups / 512.0), rest = workgroups - 512.0 * rounds;
		double us = pace.launch + rounds * (pace.round + pace.shared * steps);
		if (rest > 0.0)
			us += pace.round + (rest <= 256.0 ? pace.alone : pace.shared) * steps;
		return us;
	}

	/* Tile and number of wavefronts by the estimates above.  Where the lines lie: 1 wavefront for thousands of tiles with a short k
	 * (bf16 1x1, 107632 pixels, one stage: 13.8 us against 20.0 with four), 64 x 64 tiles where they alone fill the chip (bf16 256 ->
	 * 256 on 3800 pixels: 13.8 us against 19.2), 8 wavefronts for few tiles and a long k (fp32, 40 tiles, 325 stages: 56 us against
	 * 68), otherwise 4.  Tiles of 16 x 16 where those of 32 x 32 are few: from some 300 (five stages: 600) on those load less, 10.1 against 10.8 us for bf16 128 -> 128 3x3 with 572. */
	inline SmallPlan conv_small_plan(const avhipConvShape &s, int element_bytes)
	{
		const int64_t pixels = static_cast<int64_t>(s.N) * s.Ho * s.Wo;
		const int64_t stages = (static_cast<int64_t>(s.R) * s.S * ((static_cast<int64_t>(s.C) * element_bytes + 15) / 16) + 7) >> 3;
		SmallPlan best = { 0, 0, 0.0, 0.0, 0, 0.0 };
		int64_t tiles_16 = 0;
		const int64_t row = static_cast<int64_t>(s.C) * element_bytes;
		/* Rows of dwords or elements: two loads and a shift for a piece of elements, and bits to be cut off.  Of tiles of 16 x 16 a stage takes 1.5 and 1.9 times as long (83 layers, 6 to 16 %): with
		 * these factors the 62 that small tiles had before are 1.22 times as fast, none slower by more than 1 %. */
		const double by_rows = row % 16 == 0 ? 1.0 : row % 4 == 0 ? 1.5 : 1.9;
		/* and where rows are no whole lines of 128 bytes in 16 and 8 bits the 128 bytes of a load lie in two of them: 1.2 times (1.15 to 1.25 over 560 layers; larger tiles, which load half as much for a product, are not slower for it) */
		const double across_lines = element_bytes < 4 && row % 16 == 0 && row % 128 != 0 && row >= 64 ? 1.2 : 1.0;
		for (int i = row == 16 ? 4 : 0; i < 7; i++) /* (one chunk a tap: only the tiles of 16 x 16 count taps so) */
		{
			const int bits = PLANS[i].side_bits, side = 1 << bits, waves = 1 << PLANS[i].wave_bits;
			const Pace &pace = element_bytes == 4 ? PACE_32[i] : PACE_16[i];
			const int64_t tiles = ((pixels + side - 1) >> bits) * ((static_cast<int64_t>(s.K) + side - 1) >> bits);
			/* (beyond four tiles of 16 x 16 to a compute unit, whose wavefronts fill it, one more takes its whole time where k is long) */
			const double per_cu = tiles <= 1024 || (side == 16 && element_bytes < 4 && stages >= 12) ? static_cast<double>((tiles + 255) >> 8) : static_cast<double>(tiles) / 256.0;
			const double slower = side == 16 ? by_rows : 1.0, across = side == 16 ? across_lines : 1.0;
			const double alone = static_cast<double>((stages + waves - 1) >> PLANS[i].wave_bits) * pace.chain * slower, shared = per_cu * static_cast<double>(stages) * pace.stage * slower * across;
			const double us = (pace.launch + (element_bytes == 4 || side == 16 ? std::sqrt(alone * alone + shared * shared) : std::max(alone, shared)) + per_cu * pace.tile)
					* (side != 16 && row % 4 != 0 ? 1.25 : 1.0);
			if (side == 16)
			{
				if (best.waves_16 == 0 || us < best.us_16)
				{
					best.waves_16 = waves;
					best.us_16 = us;
				}
				tiles_16 = tiles;
			}
			else if (best.side == 0 || us < best.us)
			{
				best.side = side;
				best.waves = waves;
				best.us = best.larger_us = us;
			}
		}
		if (best.side == 0 || best.us_16 < margin_16(element_bytes, row % 128 == 0, tiles_16, stages) * best.us)
			best = best.of_16();
		return best;
	}
}

#endif /* AVHIP_CONV_ESTIMATES_HPP_ */

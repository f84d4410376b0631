/*
 * conv_ring.hip -- implicit-GEMM convolution whose operands stream through a ring of LDS buffers, for 16-bit and 8-bit layers.
 *
 * The GEMM (rows = output pixels, columns = filters, k = the 16-byte chunks of all taps in a row, 128 bytes a stage) in tiles of 256 x 128 to
 * 64 x 64.  Every operand row of a stage goes from memory straight into LDS (buffer_load ... lds: no registers, so two or three stages
 * are in flight), once per workgroup; chunks that do not exist (outside the image, behind the last one) are written as zeros by the
 * hardware.  A row of 128 bytes lies in LDS as it was loaded, but each lane chooses which chunk it loads: chunk c of row r lies in column
 * c ^ (r / 2) % 8, and then the 32 rows that a wavefront reads at once are conflict-free.
 *
 * What bounds it: with tiles of 256 x 128 the matrix cores for two thirds of the time (a stage takes 0.63 us, its products 0.49 at the 2.1 GHz that
 * these loads leave), with smaller ones the 64 bytes a clock that a compute unit loads; around the loop 3 to 6 us of first loads and results.
 * Loads in a row behind the barrier stalled their wavefronts in the queue of the memory pipeline; one by one between the products they
 * do not (a 64 x 64 tile with a compute unit to itself: 0.24 -> 0.21 us a stage, 256 x 128: 38.7 -> 34.3 us on the second layer below).
 * Measured, before (the kernel that took the layer then: gather, image tiles or small tiles) and now: bf16 192 -> 384 3x3 stride 2 on 25 images of 58 x 58 and its
 * 1x1 384 -> 768 73 -> 56 us, fp16 224 -> 112 3x3 on 79 x 26 x 26 with an ELU 54 -> 43.5 (with LINEAR or
 * RELU the estimates keep it in image tiles, 49), int8 144 -> 80 3x3 on 81 x 39 x 39 43.5 -> 27, bf16 256 -> 512 3x3 stride 2
 * on 23 x 35 x 35 34 -> 21, bf16 192 -> 384 3x3 stride 2 on 11 x 41 x 41 15.3 -> 11.5.
 * Activations by a call: a work-item's sixteen results of a tile at once, residual requested ahead (ACT_VECTORS; four at a time in a loop before): f16 32 -> 448 3x3 on 234 x 12 x 12 with
 * a residual and an ELU 43.3 -> 35.8 us, bf16 488 -> 320 1x1 stride 2 on 22 x 54 x 55 with an ELU 21.3 -> 16.8, with a sigmoid 21.4 -> 18.8, 65 such layers 1.02 to 1.37 times as fast, 1.11 on average.
 */
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "conv_ring.hpp"
#include "conv_ring_plan.hpp"
#include "conv_small.hpp"
#include "mfma_core.hpp"

namespace
{
	using namespace avhip;

	struct RingGeom
	{
		int H, W, C, K, R, S, Ho, Wo, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, flip;
		int chunks_per_tap; /* 16-byte chunks of the channels of one tap */
		unsigned int by_chunks, by_s; /* ceil(2^32 / chunks_per_tap), ceil(2^16 / S): division by multiplication */
		int pixels, images;
		unsigned int pixel_tiles, filter_tiles;
		Divisor by_wo, by_ho, by_tiles; /* by_tiles: of the faster of the two */
		int pixels_first; /* order of the tiles: pixel tiles run fastest within an XCD (more weights than image), or filter tiles */
	};

	/* LDS accesses of a wavefront to its own part stay in this order (the hardware does them in order, without a barrier) */
	__device__ __forceinline__ void wave_order()
	{
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	}
	/* at most N vector-memory operations and no LDS operation of this wavefront in flight, then the barrier */
	template<int N>
	__device__ __forceinline__ void wait_and_meet()
	{
		asm volatile("" ::: "memory");
		__builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 7 << 4);
		__builtin_amdgcn_s_barrier();
		asm volatile("" ::: "memory");
	}
	typedef __attribute__((address_space(3))) void *lds_ptr;

	/* WP x WF wavefronts of TP x TF MFMA tiles of 32 x 32 (pixels x filters), DEPTH buffers */
	template<typename TE, typename Epi, int WP, int WF, int TP, int TF, int DEPTH, int PER_SIMD, int ACT>
	__global__ __launch_bounds__(64 * WP * WF, PER_SIMD) void k_conv_ring(const TE *__restrict__ x, const TE *__restrict__ w, RingGeom g, Epi epi)
	{
		constexpr unsigned int SZ = sizeof(TE);
		constexpr int WAVES = WP * WF, PX = 32 * WP * TP, FT = 32 * WF * TF;
		constexpr int X_LOADS = PX / 8 / WAVES, W_LOADS = FT / 8 / WAVES, LOADS = X_LOADS + W_LOADS; /* of a wavefront and stage, 8 rows of 128 bytes each */
		static_assert(WAVES % 2 == 0 && PX % (8 * WAVES) == 0 && FT % (8 * WAVES) == 0, "whole loads, of rows of one parity per wavefront");
		static_assert(DEPTH >= 2 && DEPTH <= 4, "buffers");
		constexpr int SLOT = (PX + FT) * 128;
		static_assert(2 * SLOT >= WAVES * 4096, "a tile of results per wavefront");
		constexpr bool VEC = ACT != ACT_ANY;
		typedef typename Epi::scalar_t scalar_t;
		typedef Pack<scalar_t, 4> quad_t;
		/* arrays of their own: the compiler tells the loads into one buffer from the reads of another */
		__shared__ __attribute__((aligned(16))) char ring0[SLOT];
		__shared__ __attribute__((aligned(16))) char ring1[SLOT];
		__shared__ __attribute__((aligned(16))) char ring2[DEPTH > 2 ? SLOT : 16];
		__shared__ __attribute__((aligned(16))) char ring3[DEPTH > 3 ? SLOT : 16];
		__shared__ uint2 pixel[PX];

		const int lane = threadIdx.x & 63;
		const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
		const unsigned int t = xcd_block(blockIdx.y * g.pixel_tiles + blockIdx.x, g.pixel_tiles * g.filter_tiles);
		const unsigned int slow = g.by_tiles.of(t), fast = t - slow * (g.pixels_first ? g.pixel_tiles : g.filter_tiles);
		const unsigned int pixel_tile = g.pixels_first ? fast : slow, filter_tile = g.pixels_first ? slow : fast;
		const int p0 = static_cast<int>(pixel_tile) * PX, k0 = static_cast<int>(filter_tile) * FT;

		const unsigned int c_bytes = g.C * SZ, filter_bytes = g.R * g.S * c_bytes;
		const __amdgpu_buffer_rsrc_t rx = make_buffer(x, static_cast<unsigned int>(g.images) * g.H * g.W * c_bytes);
		const __amdgpu_buffer_rsrc_t rw = make_buffer(w, static_cast<unsigned int>(g.K) * filter_bytes);

		/* origin and border mask (bit = tap inside the image) of every pixel */
		if (static_cast<int>(threadIdx.x) < PX)
		{
			const int p = p0 + static_cast<int>(threadIdx.x);
			const bool row_ok = p < g.pixels;
			const int pp = row_ok ? p : 0;
			const int line = static_cast<int>(g.by_wo.of(pp)), ow = pp - line * g.Wo;
			const int n = static_cast<int>(g.by_ho.of(line)), oh = line - n * g.Ho;
			const int ih0 = oh * g.stride_h + g.pad_h, iw0 = ow * g.stride_w + g.pad_w;
			unsigned int inside = 0;
			if (row_ok)
			{
				unsigned int cols = 0;
				for (int j = 0; j < g.S; j++)
				{
					const int iw = iw0 + (g.flip ? g.S - 1 - j : j) * g.dil_w;
					if (iw >= 0 && iw < g.W)
						cols |= 1u << j;
				}
				for (int i = 0; i < g.R; i++)
				{
					const int ih = ih0 + (g.flip ? g.R - 1 - i : i) * g.dil_h;
					if (ih >= 0 && ih < g.H)
						inside |= cols << (i * g.S);
				}
			}
			pixel[threadIdx.x] = make_uint2(static_cast<unsigned int>((n * g.H + ih0) * g.W + iw0) * c_bytes, inside);
		}
		static_assert(PX <= 64 * WAVES, "one pixel per work-item");
		__syncthreads();
		/* this lane loads 16 bytes of the rows 8 (wave + WAVES i) + lane / 8; chunk c of row r lies in column c ^ (r / 2) % 8 of its buffer, so it is
		 * the lane that chooses which chunk it loads */
		const int load_row = 8 * wave + (lane >> 3);
		uint2 origin[X_LOADS];
#pragma unroll
		for (int i = 0; i < X_LOADS; i++)
			origin[i] = pixel[8 * WAVES * i + load_row];
		const unsigned int w_origin = static_cast<unsigned int>(k0 + load_row) * filter_bytes; /* filters past the last lie outside the buffer */
		const unsigned int chunks = g.R * g.S * g.chunks_per_tap;
		unsigned int chunk = (lane & 7) ^ (lane >> 4) ^ ((wave & 1) << 2);
		/* where the loads of the next stage to be requested come from: worked out ahead, among products */
		unsigned int x_from[X_LOADS], w_from[W_LOADS];
		auto prepare = [&]() __attribute__((always_inline))
		{
			const bool live = chunk < chunks;
			const unsigned int tap = __umulhi(chunk, g.by_chunks);
			const unsigned int c = chunk - tap * g.chunks_per_tap;
			const unsigned int ti = (tap * g.by_s) >> 16, tj = tap - ti * g.S;
			const unsigned int i = g.flip ? g.R - 1 - ti : ti, j = g.flip ? g.S - 1 - tj : tj;
			const unsigned int x_tap = ((i * g.dil_h) * g.W + j * g.dil_w) * c_bytes + 16 * c;
			const unsigned int bit = live ? 1u << (tap & 31) : 0u;
			const unsigned int w_at = w_origin + 16 * chunk;
			chunk += 8;
#pragma unroll
			for (int q = 0; q < X_LOADS; q++)
				x_from[q] = (origin[q].y & bit) ? origin[q].x + x_tap : OUT_OF_RANGE;
#pragma unroll
			for (int q = 0; q < W_LOADS; q++)
				w_from[q] = live ? w_at + 8 * WAVES * q * filter_bytes : OUT_OF_RANGE;
		};
		auto load = [&](char *slot, int q) __attribute__((always_inline))
		{
			if (q < X_LOADS)
				__builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(slot + (wave + WAVES * q) * 1024), 16, static_cast<int>(x_from[q]), 0, 0, 0);
			else
				__builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)(slot + PX * 128 + (wave + WAVES * (q - X_LOADS)) * 1024), 16,
						static_cast<int>(w_from[q - X_LOADS]), 0, 0, 0);
		};
		auto issue = [&](char *slot) __attribute__((always_inline))
		{
#pragma unroll
			for (int q = 0; q < LOADS; q++)
				load(slot, q);
		};

		const int wp = wave / WF, wf = wave - wp * WF;
		const int r = lane & 31, half = lane >> 5;
		typename Mma<TE>::acc_t acc[TF][TP]; /* [filters][pixels] */
#pragma unroll
		for (int i = 0; i < TF; i++)
#pragma unroll
			for (int j = 0; j < TP; j++)
#pragma unroll
				for (int v = 0; v < 16; v++)
					acc[i][j][v] = 0;
		const int x_row = (wp * TP * 32 + r) * 128, w_row = PX * 128 + (wf * TF * 32 + r) * 128;
		Chunk cx[2][TP], cw[2][TF];
		auto read = [&](const char *slot, int slab) __attribute__((always_inline))
		{
			const int column = 16 * ((2 * slab + half) ^ ((r >> 1) & 7));
#pragma unroll
			for (int j = 0; j < TP; j++)
				cx[slab & 1][j].u = *reinterpret_cast<const uint4*>(slot + x_row + 4096 * j + column);
#pragma unroll
			for (int i = 0; i < TF; i++)
				cw[slab & 1][i].u = *reinterpret_cast<const uint4*>(slot + w_row + 4096 * i + column);
		};
		auto multiply = [&](int slab) __attribute__((always_inline))
		{
#pragma unroll
			for (int i = 0; i < TF; i++)
#pragma unroll
				for (int j = 0; j < TP; j++)
					Mma<TE>::run(cw[slab & 1][i], cx[slab & 1][j], acc[i][j]);
		};

		/* what the epilogue needs of the filters */
		const int quad = lane & 7;
		typename Epi::Columns columns[TF];
#pragma unroll
		for (int i = 0; i < TF; i++)
			epi.load_columns(k0 + (wf * TF + i) * 32 + 4 * quad, columns[i]);

		prepare();
		issue(ring0);
		prepare();
		if (DEPTH > 2)
		{
			issue(ring1);
			prepare();
		}
		if (DEPTH > 3)
		{
			issue(ring2);
			prepare();
		}
		const int stages = static_cast<int>((chunks + 7) / 8), rest = stages % DEPTH;
		/* One stage.  All of its operands are in registers before its last products, so the buffer changes hands there: behind the barrier the next
		 * stage has arrived and its first operands are read while those products run.  The loads into the buffer that became free that way a stage
		 * ago go out one by one between products: in a row they fill the queue of the memory pipeline and the wavefront stands. */
		auto step = [&](const char *now, const char *next, char *free) __attribute__((always_inline))
		{
#pragma unroll
			for (int slab = 0; slab < 3; slab++)
			{
				read(now, slab + 1);
				__builtin_amdgcn_sched_barrier(0);
#pragma unroll
				for (int q = 0; q < LOADS; q++)
					if (q * 3 / LOADS == slab)
						load(free, q);
				__builtin_amdgcn_sched_barrier(0);
				multiply(slab);
				__builtin_amdgcn_sched_barrier(0);
			}
			wait_and_meet<(DEPTH - 2) * LOADS>();
			__builtin_amdgcn_sched_barrier(0);
			read(next, 0);
			__builtin_amdgcn_sched_barrier(0);
			multiply(3);
			prepare();
		};
		wait_and_meet<(DEPTH - 2) * LOADS>();
		read(ring0, 0);
		/* (no way out of the loop but its end: past one, the compiler waits for all loads in every round) */
		for (int round = stages / DEPTH; round > 0; round--)
		{
			step(ring0, ring1, DEPTH == 2 ? ring1 : DEPTH == 3 ? ring2 : ring3);
			step(ring1, DEPTH == 2 ? ring0 : ring2, ring0);
			if (DEPTH > 2)
				step(ring2, DEPTH == 3 ? ring0 : ring3, ring1);
			if (DEPTH > 3)
				step(ring3, ring0, ring2);
		}
		if (rest > 0)
			step(ring0, ring1, DEPTH == 2 ? ring1 : DEPTH == 3 ? ring2 : ring3);
		if (DEPTH > 2 && rest > 1)
			step(ring1, ring2, ring0);
		if (DEPTH > 3 && rest > 2)
			step(ring2, ring3, ring1);
		wait_and_meet<0>();

		/* A lane holds, of pixel r of each pixel tile, the filters 8 v + 4 half .. + 3 of each filter tile.  Tile by tile through four kilobytes of the
		 * wavefront's own: runs of four filters in the order (run, pixel ^ 2 run), conflict-free both ways; then eight lanes have a pixel. */
		constexpr int IN_ONE = SLOT / 4096 < WAVES ? SLOT / 4096 : WAVES;
		quad_t *mine = reinterpret_cast<quad_t*>(wave < IN_ONE ? ring0 + wave * 4096 : ring1 + (wave - IN_ONE) * 4096);
		const int pass_row = lane >> 3;
		auto row_of = [&](int j, int pass) __attribute__((always_inline))
		{
			return p0 + (wp * TP + j) * 32 + 8 * pass + pass_row;
		};
		typename Epi::template Residual<4> residual[2][4];
		auto request = [&](int tile) __attribute__((always_inline))
		{
			const int i = tile / TP, j = tile - i * TP, k = k0 + (wf * TF + i) * 32 + 4 * quad;
#pragma unroll
			for (int pass = 0; pass < 4; pass++)
				if (row_of(j, pass) < g.pixels && k < g.K)
					epi.template load_residual<4>(static_cast<int64_t>(row_of(j, pass)) * g.K + k, residual[tile & 1][pass]);
		};
		if (VEC)
			request(0);
#pragma unroll
		for (int tile = 0; tile < TP * TF; tile++)
		{
			const int i = tile / TP, j = tile - i * TP, k = k0 + (wf * TF + i) * 32 + 4 * quad;
#pragma unroll
			for (int v = 0; v < 4; v++)
			{
				quad_t q;
#pragma unroll
				for (int e = 0; e < 4; e++)
					q.v[e] = acc[i][j][4 * v + e];
				mine[(2 * v + half) * 32 + (r ^ (2 * (2 * v + half)))] = q;
			}
			wave_order();
			auto hand_over = [&](int pass) __attribute__((always_inline))
			{
				const quad_t v = mine[quad * 32 + ((8 * pass + pass_row) ^ (2 * quad))];
				if (row_of(j, pass) < g.pixels && k < g.K)
					epi.template store_at<ACT, VEC, 4>(static_cast<int64_t>(row_of(j, pass)) * g.K + k, k, v.v, columns[i], VEC ? &residual[tile & 1][VEC ? pass : 0] : nullptr);
			};
			if constexpr (ACT == ACT_VECTORS)
			{
				if (tile + 1 < TP * TF)
					request(tile + 1);
				float v[4][4];
#pragma unroll
				for (int pass = 0; pass < 4; pass++)
				{
					const quad_t q = mine[quad * 32 + ((8 * pass + pass_row) ^ (2 * quad))];
#pragma unroll
					for (int e = 0; e < 4; e++)
						v[pass][e] = q.v[e];
				}
				epi.store_runs(k, v, columns[i], residual[tile & 1], [&](int pass, int64_t &idx) __attribute__((always_inline))
				{
					idx = static_cast<int64_t>(row_of(j, pass)) * g.K + k;
					return row_of(j, pass) < g.pixels && k < g.K;
				});
			}
			else if constexpr (VEC)
			{
				if (tile + 1 < TP * TF)
					request(tile + 1);
#pragma unroll
				for (int pass = 0; pass < 4; pass++)
					hand_over(pass);
			}
			else
			{
#pragma unroll 1 /* the switch over the activations once per tile */
				for (int pass = 0; pass < 4; pass++)
					hand_over(pass);
			}
			wave_order();
		}
	}
}

namespace
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

	/* no layer is estimated below a workgroup of the fastest pace, beginning and end */
	constexpr double ring_at_least_us(double stages)
	{
		double fixed = RING_PLANS[0].launch + RING_PLANS[0].tile, stage = RING_PLANS[0].stage;
		for (const RingPlan &p : RING_PLANS)
		{
			fixed = p.launch + p.tile < fixed ? p.launch + p.tile : fixed;
			stage = p.stage < stage ? p.stage : stage;
		}
		return fixed + stage * stages;
	}

	struct RingChoice
	{
		int plan;
		double us;
	};
	RingChoice ring_choice(const avhipConvShape &s, double stages, int out_bytes, HandOver hand_over, bool residual)
	{
		const double pixels = static_cast<double>(s.N) * s.Ho * s.Wo;
		const double megabytes = pixels * s.K * out_bytes * (residual ? 2.0e-6 : 1.0e-6);
		RingChoice best = { -1, 0.0 };
		for (int i = 0; i < 4; i++)
		{
			const RingPlan &p = RING_PLANS[i];
			const double tile = p.tile + (hand_over == HandOver::ELEMENTS ? p.elements : hand_over == HandOver::ACTIVATION ? p.activation : 0.0);
			const double loads = std::ceil(pixels / p.pixels) * ((s.K + p.filters - 1) / p.filters) / 256.0; /* of workgroups, one per compute unit each */
			const double rounds = std::floor(loads / p.per_cu), rest = std::ceil(loads - rounds * p.per_cu);
			const double us = p.launch + (rounds + (rest > 0.0 ? 1.0 : 0.0)) * tile + (rounds * p.per_cu + rest) * p.stage * stages + p.megabyte * megabytes;
			if (best.plan < 0 || us < best.us)
				best = { i, us };
		}
		return best;
	}

	/* The tile that the layer gets and its estimate, or no plan where it is left to the other kernels */
	RingChoice ring_route(const avhipConvShape &s, int element_bytes, int out_bytes, const SmallChoice &small, bool residual)
	{
		const RingChoice none = { -1, 0.0 };
		/* layers that the few-channel kernels have taken before this one is asked */
		if (small.hand_over == HandOver::PLAIN && conv_few_channels(s, element_bytes))
			return none;
		/* (the switch of the small tiles is this kernel's too: at 0 the kernels with fixed tiles of 128 x 128 are asked for, below it small ones) */
		if (element_bytes > 2 || static_cast<int64_t>(s.C) * element_bytes % 16 != 0 || s.C * element_bytes < 32 || !conv_small_possible(s, element_bytes) || conv_small_threshold() <= 0)
			return none;
		/* of 8-bit one-tap layers the persistent kernels are a fifth to a third faster than they are estimated (17 layers) */
		if (element_bytes == 1 && small.one_tap_us > 0.0)
			return none;
		/* 15 % below the others' estimates, which are the coarser ones (those of image tiles and one-tap kernels up to 1.9 and 1.7 times too low where filters fill no
		 * blocks of 64 or channels no 128 bytes: 32 -> 440 3x3 on 4 x 61 x 64 takes 19.6 us there against 13.2 here, and stays there): of the
		 * 410 layers one is then slower than before (bf16, a filter count that is no multiple of four), and the mean gain is 11.7 of the 13.9 % that the best choice for each would have */
		/* Small tiles of fewer than 32 filters of a 16-bit layer take down to three quarters of their estimate, which counts the filters that do not exist as loaded.
		 * Of 140 layers of 8 to 64 filters 32 leave the ring for that, 15 of them 2 to 24 % slower in it (fp16 512 -> 13 1x1 on 187 x 10 x 11 7.7 : 10.2 us, bf16 400 -> 10
		 * 3x3 on 94 x 30 x 30 58 : 70.5), the others 11 % faster at most; of 70 that the rule was not made from 32, 0.70 to 1.16 times as fast in
		 * it and 0.97 on average, where the 38 that stay are 1.10 times as fast.  8-bit layers stay (25 of them 1.02 times as fast in the ring). */
		const double others = element_bytes == 2 && small.larger_preferred && s.K < 32 ? (0.75 + 0.25 / 32.0 * s.K) * small.larger_us : small.larger_us;
		const double limit = 0.85 * others, stages = std::ceil(static_cast<double>(s.R) * s.S * (s.C * element_bytes / 16) / 8.0);
		/* one workgroup takes longer than that, whatever its tile: the smallest layers, whose calls cost the host no less than the GPU */
		if (ring_at_least_us(stages) >= limit)
			return none;
		const RingChoice choice = ring_choice(s, stages, out_bytes, small.hand_over, residual);
		if (choice.us >= limit)
			return none;
		/* Tiles of 16 x 16 take a layer from here where they are estimated at 0.69 of its time or less.  Both estimates are loose where this one is low (5 to 12 %, and 64 x 64 tiles alone on a compute unit take longer
		 * than theirs): at 1.0 of it bf16 192 -> 192 3x3 on 14 x 11 x 11 moved the wrong way, 9.6 -> 11.5 us; what lies between stays where it was timed. */
		return small.preferred && small.plan.side == 16 && small.us < 0.69 * choice.us ? none : choice;
	}
}

namespace avhip
{
	double conv_ring_us(const avhipConvShape &s, int element_bytes, int out_bytes, const SmallChoice &small, bool residual)
	{
		return ring_route(s, element_bytes, out_bytes, small, residual).us;
	}

	template<typename TE, typename Epi>
	bool conv_ring_launch(hipStream_t stream, const avhipConvShape &s, const void *x, const void *w, const Epi &epi, const SmallChoice &small)
	{
		constexpr int SZ = static_cast<int>(sizeof(TE));
		const int64_t pixels = static_cast<int64_t>(s.N) * s.Ho * s.Wo;
		const bool simple = small.hand_over == HandOver::PLAIN;
		const int plan = ring_route(s, SZ, Epi::out_bytes, small, epi.z != nullptr).plan;
		if (plan < 0 || in_place(s, x, SZ, epi.y, Epi::out_bytes))
			return false;
		const int px = RING_PLANS[plan].pixels, ft = RING_PLANS[plan].filters;
		const int64_t pixel_tiles = (pixels + px - 1) / px, filter_tiles = (static_cast<int64_t>(s.K) + ft - 1) / ft;
		if (pixel_tiles * 512 >= (1ll << 32) /* work-items of a launch along one direction */ || filter_tiles > 65535 || pixel_tiles * filter_tiles > 0x7FFFFFFFll || pixels >= (1ll << 31) - 256)
			return false;
		RingGeom g;
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
		g.chunks_per_tap = (s.C * SZ + 15) / 16;
		g.by_chunks = static_cast<unsigned int>(((1ll << 32) + g.chunks_per_tap - 1) / g.chunks_per_tap);
		g.by_s = (65536 + s.S - 1) / s.S;
		g.pixels = static_cast<int>(pixels);
		g.images = s.N;
		g.pixels_first = static_cast<int64_t>(s.K) * s.R * s.S > static_cast<int64_t>(s.N) * s.H * s.W ? 1 : 0;
		g.pixel_tiles = static_cast<unsigned int>(pixel_tiles);
		g.filter_tiles = static_cast<unsigned int>(filter_tiles);
		g.by_wo = divisor(s.Wo);
		g.by_ho = divisor(s.Ho);
		g.by_tiles = divisor(g.pixels_first ? g.pixel_tiles : g.filter_tiles);
		const dim3 grid(g.pixel_tiles, g.filter_tiles);
#define AVHIP_RING(WP, WF, TP, TF, DEPTH, PER_SIMD) \
		do \
		{ \
			if (simple) \
				hipLaunchKernelGGL((k_conv_ring<TE, Epi, WP, WF, TP, TF, DEPTH, PER_SIMD, ACT_SIMPLE>), grid, dim3(64 * WP * WF), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi); \
			else if (Epi::runs && epi.vec && small.hand_over == HandOver::ACTIVATION) \
				hipLaunchKernelGGL((k_conv_ring<TE, Epi, WP, WF, TP, TF, DEPTH, PER_SIMD, Epi::runs ? ACT_VECTORS : ACT_ANY>), grid, dim3(64 * WP * WF), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi); \
			else \
				hipLaunchKernelGGL((k_conv_ring<TE, Epi, WP, WF, TP, TF, DEPTH, PER_SIMD, ACT_ANY>), grid, dim3(64 * WP * WF), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi); \
		} while (0)
		switch (plan)
		{
			case 0:
				AVHIP_RING(4, 2, 2, 2, 3, 2);
				break;
			case 1:
				AVHIP_RING(4, 2, 1, 2, 4, 2);
				break;
			case 2:
				AVHIP_RING(4, 2, 1, 1, 3, 4);
				break;
			default:
				AVHIP_RING(2, 2, 1, 1, 3, 3);
				break;
		}
#undef AVHIP_RING
		return true;
	}

#define AVHIP_INSTANTIATE(TE, EPI) template bool conv_ring_launch<TE, EPI>(hipStream_t, const avhipConvShape&, const void*, const void*, const EPI&, const SmallChoice&);
	AVHIP_INSTANTIATE(f16_t, FloatEpilogue<f16_t>)
	AVHIP_INSTANTIATE(bf16_t, FloatEpilogue<bf16_t>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_EXACT>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_REQUANT>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_FLOAT_I32>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_FLOAT_I8>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_FLOAT_F32>)
#undef AVHIP_INSTANTIATE
}

namespace
{
	/* as the launcher asks for a call with this epilogue, tensors at address 16 */
	template<typename TE, typename Epi>
	RingChoice route_of_call(const avhipConvShape &s, int hand_over, int residual)
	{
		Epi epi { };
		epi.vec = hand_over == 0;
		epi.activation = hand_over == 2 ? ACT_ELU : ACT_LINEAR;
		if (residual != 0)
			epi.z = reinterpret_cast<decltype(epi.z)>(16);
		return ring_route(s, static_cast<int>(sizeof(TE)), Epi::out_bytes, conv_small_choice<TE>(s, epi), residual != 0);
	}
	RingChoice route_of_call(int x_dtype, int y_dtype, const avhipConvShape *shape, int hand_over, int residual)
	{
		if (shape == nullptr || hand_over < 0 || hand_over > 2)
			return { -1, 0.0 };
		switch (x_dtype)
		{
			case DT_FLOAT16:
				return route_of_call<f16_t, FloatEpilogue<f16_t>>(*shape, hand_over, residual);
			case DT_BFLOAT16:
				return route_of_call<bf16_t, FloatEpilogue<bf16_t>>(*shape, hand_over, residual);
			case DT_INT8:
				if (y_dtype == DT_INT8)
					return route_of_call<int8_t, Int8Epilogue<I8_REQUANT>>(*shape, hand_over, residual);
				if (y_dtype == DT_INT32)
					return route_of_call<int8_t, Int8Epilogue<I8_EXACT>>(*shape, hand_over, residual);
				return route_of_call<int8_t, Int8Epilogue<I8_FLOAT_F32>>(*shape, hand_over, residual);
			default:
				return { -1, 0.0 };
		}
	}
}

extern "C" double avhip_conv2d_ring_us(int x_dtype, int y_dtype, const avhipConvShape *shape, int hand_over, int residual)
{
	return route_of_call(x_dtype, y_dtype, shape, hand_over, residual).us;
}

extern "C" int avhip_conv2d_ring_plan(int x_dtype, int y_dtype, const avhipConvShape *shape, int hand_over, int residual)
{
	return route_of_call(x_dtype, y_dtype, shape, hand_over, residual).plan;
}

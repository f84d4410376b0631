/*
 * conv_small.hip -- implicit-GEMM convolution for problems that do not fill the chip with 128 x 128 workgroup tiles.
 *
 * The GEMM (rows = output pixels, columns = filters, k = (tap, channel)) is cut into tiles of 32 x 32 or 64 x 64 (of 16 x 16: conv_small16.hip) and the k range
 * of a tile is shared by the one, four or eight wavefronts of a workgroup, so that a layer of a few hundred pixels still occupies
 * the chip; the partial tiles are added through LDS in a fixed order.  There is no barrier in the k loop: each wavefront loads its
 * own operands, 128 bytes of k of every row at a time, eight lanes to a row, and brings them into MFMA layout through its own
 * part of LDS.  k runs over the 16-byte chunks of all taps in a row, so channel counts that are no multiple of 64 cost nothing.
 * Where the channels of a tap are no whole number of chunks the last chunk of a tap is cut off in registers, and 16-bit or 8-bit
 * rows that start between two dwords are loaded as the dwords around them and shifted.
 *
 * fp32 with 64 x 64: products of bf16 pieces (struct Pieces of mfma_core.hpp), cut by the wavefront that multiplies; with 32 x 32 the cutting takes as long as the
 * products save.  96 -> 64 5x5 on 21 images of 57 x 53 287 -> 131 us (image tiles before), 352 -> 112 3x3 stride 2 on 76 of 35 x 35 with an ELU 235 -> 169 (32 x 32).
 *
 * What bounds it: the 64 bytes per clock that a compute unit loads (128 clocks per stage of a 32 x 32 tile, 256 per stage of a
 * 64 x 64 tile, which needs half as much per product), for fp32 the matrix cores, and for the smallest problems the latency of
 * one launch.  Operands loaded straight in MFMA layout (32 lines per load instruction) took 55 to 60 clocks a kilobyte here, by
 * rows 20.  Measured, before (that form, 128 x 128 gather kernel where it was preferred) and now: bf16 128 -> 128 3x3 on 2912
 * pixels 11.8 -> 7.6 us, 256 -> 256 3x3 on 3800 pixels 17.3 -> 12.7 us, fp32 64 -> 218 5x5 on 1568 pixels 121 -> 23 us, fp16 72 -> 100
 * channels 3x3 with an ELU and a residual on 13520 pixels 31.8 -> 12.9 us, int8 128 -> 128 stride 2 on 6720 pixels 21.7 -> 9.8 us.  Against the general
 * gather kernel, element by element: fp16 185 -> 160 3x3 on 8640 pixels 157 -> 25 us, fp16 370 -> 64 3x3 on 57876 pixels 414 -> 66 us,
 * fp32 395 -> 32 5x5 stride 2 on 1170 pixels 1068 -> 62 us, bf16 90 -> 256 1x1 on 627200 pixels 495 -> 214 us.
 */
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "conv_small.hpp"
#include "conv_small_rows.hpp"
#include "mfma_core.hpp"

namespace
{
	using namespace avhip;

	/* LDS accesses of a wavefront to its own part stay in this order (the hardware does them in order, without a barrier) */
	__device__ __forceinline__ void wave_order()
	{
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	}

	/* T x T MFMA tiles of 32 x 32 per wavefront, KW wavefronts on one tile. */
	template<typename TE, typename Epi, int T, int KW, int ACT, int ROW = ROWS_OF_CHUNKS>
	__global__ __launch_bounds__(64 * KW, KW == 8 ? 2 : T == 1 ? 3 : 2) void k_conv_small(const TE *__restrict__ x, const TE *__restrict__ w, SmallGeom g, Epi epi)
	{
		constexpr unsigned int SZ = sizeof(TE);
		constexpr int SIDE = 32 * T;
		constexpr int LOADS = 4 * T; /* loads of 8 rows each, per operand and stage */
		constexpr int QUADS = SIDE / 4; /* runs of four filters of a pixel */
		constexpr int PITCH = T == 1 ? SIDE + 2 : SIDE + 1; /* 16-byte slots between two runs of a pixel: conflict-free both ways */
		constexpr int SLOTS = QUADS * PITCH > 2 * SIDE * 8 ? QUADS * PITCH : 2 * SIDE * 8;
		constexpr int DEPTH = T == 1 ? 2 : 1; /* stages in flight */
		constexpr bool VEC = ACT != ACT_ANY;
		constexpr bool BY_PIECES = std::is_same<TE, float>::value && T == 2; /* (with 32 x 32 the cutting costs what the products save) */
		typedef typename Epi::scalar_t scalar_t;
		typedef Pack<scalar_t, 4> quad_t;
		/* each wavefront its own part: rows of the stage being multiplied, then its partial tile */
		__shared__ __attribute__((aligned(16))) uint4 lds[KW][SLOTS];

		const int lane = threadIdx.x & 63;
		const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
		uint4 *mine = lds[wave];
		/* Each XCD gets a contiguous run of the tiles, and within it the tiles that share the larger operand are neighbours, so
		 * that its L2 fetches that operand once. */
		const unsigned int t = xcd_block(blockIdx.y * g.pixel_tiles + blockIdx.x, g.pixel_tiles * g.filter_tiles);
		const unsigned int slow = g.by_tiles.of(t), fast = t - slow * (g.pixels_first ? g.pixel_tiles : g.filter_tiles);
		const unsigned int pixel_tile = g.pixels_first ? fast : slow, filter_tile = g.pixels_first ? slow : fast;
		const int p0 = static_cast<int>(pixel_tile) * SIDE, k0 = static_cast<int>(filter_tile) * SIDE;

		const unsigned int c_bytes = g.C * SZ, filter_bytes = g.R * g.S * c_bytes;
		const __amdgpu_buffer_rsrc_t rx = make_buffer(x, (static_cast<unsigned int>(g.images) * g.H * g.W * c_bytes + 3) & ~3u); /* a dword never crosses a page */
		const __amdgpu_buffer_rsrc_t rw = make_buffer(w, (static_cast<unsigned int>(g.K) * filter_bytes + 3) & ~3u);

		/* origin and border mask (bit = tap inside the image) of one pixel per lane, handed through LDS to the lanes that load it */
		uint2 *pixel = reinterpret_cast<uint2*>(mine);
		if (T == 2 || lane < SIDE)
		{
			const int p = p0 + lane;
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
			pixel[lane] = make_uint2(static_cast<unsigned int>((n * g.H + ih0) * g.W + iw0) * c_bytes, inside);
		}
		wave_order();
		/* this lane loads chunk (lane % 8) of the rows 8 i + lane / 8: eight lanes read the 128 bytes of a row together */
		const int load_row = lane >> 3, load_chunk = lane & 7;
		uint2 origin[LOADS];
#pragma unroll
		for (int i = 0; i < LOADS; i++)
			origin[i] = pixel[8 * i + load_row];
		wave_order();
		const unsigned int w_origin = static_cast<unsigned int>(k0 + load_row) * filter_bytes; /* filters past the last lie outside the buffer */

		typename Mma<TE>::acc_t acc[T][T]; /* [filters][pixels] */
		/* k = the 16-byte chunks of (tap, channel) in a row, eight a stage; each wavefront takes a contiguous share of the stages */
		const int chunks = g.R * g.S * g.chunks_per_tap;
		const int stages = (chunks + 7) / 8;
		const int share = (stages + KW - 1) / KW;
		const int first = wave * share;
		const int count = stages - first < share ? stages - first : share; /* may be negative: nothing left for this wavefront */
		const unsigned int chunks_mine = count > 0 ? (chunks < 8 * (first + count) ? chunks : 8 * (first + count)) : 0;
		unsigned int chunk;
		struct Stage
		{
			Piece<ROW> xs[LOADS], ws[LOADS];
			unsigned int x_tap, w_at; /* not whole chunks: where the pieces start (the lowest two bits are used) */
			int left; /* and the bytes of the row from there */
		};
		auto fetch = [&](Stage &to) __attribute__((always_inline))
		{
			const bool live = chunk < chunks_mine;
			/* (one chunk a tap: the factor would be 2^32) */
			const unsigned int tap = ROW != ROWS_OF_CHUNKS && g.chunks_per_tap == 1 ? chunk : __umulhi(chunk, g.by_chunks);
			const unsigned int c = chunk - tap * g.chunks_per_tap;
			const unsigned int ti = (tap * g.by_s) >> 16, tj = tap - ti * g.S;
			const unsigned int i = g.flip ? g.R - 1 - ti : ti, j = g.flip ? g.S - 1 - tj : tj;
			const unsigned int x_tap = ((i * g.dil_h) * g.W + j * g.dil_w) * c_bytes + 16 * c;
			const unsigned int bit = live ? 1u << (tap & 31) : 0u;
			const unsigned int w_at = w_origin + (ROW == ROWS_OF_CHUNKS ? 16 * chunk : tap * c_bytes + 16 * c);
			if (ROW != ROWS_OF_CHUNKS)
			{
				to.x_tap = x_tap;
				to.w_at = w_at;
				to.left = static_cast<int>(c_bytes - 16 * c);
			}
			chunk += 8;
#pragma unroll
			for (int q = 0; q < LOADS; q++)
				to.xs[q].fetch(rx, (origin[q].y & bit) ? origin[q].x + x_tap : OUT_OF_RANGE);
#pragma unroll
			for (int q = 0; q < LOADS; q++)
				to.ws[q].fetch(rw, live ? w_at + 8 * q * filter_bytes : OUT_OF_RANGE);
		};
		Stage stage[DEPTH];
		auto begin = [&]() __attribute__((always_inline))
		{
#pragma unroll
			for (int i = 0; i < T; i++)
#pragma unroll
				for (int j = 0; j < T; j++)
#pragma unroll
					for (int v = 0; v < 16; v++)
						acc[i][j][v] = 0;
			chunk = 8 * first + load_chunk;
#pragma unroll
			for (int d = 0; d < DEPTH; d++)
				fetch(stage[d]);
		};
		begin();

		/* what the epilogue needs is requested behind the first operands and arrives with them */
		constexpr int ROWS = 64 * KW / QUADS; /* pixels handed over in one pass of the workgroup */
		constexpr int PASSES = (SIDE + ROWS - 1) / ROWS;
		const int quad = static_cast<int>(threadIdx.x) % QUADS, row0 = static_cast<int>(threadIdx.x) / QUADS;
		const int kcol = k0 + 4 * quad;
		typename Epi::Columns columns;
		epi.load_columns(kcol, columns);
		typename Epi::template Residual<4> residual[PASSES];
		auto request_residual = [&]() __attribute__((always_inline))
		{
#pragma unroll
			for (int pass = 0; pass < PASSES; pass++)
			{
				const int row = row0 + ROWS * pass;
				if (row < SIDE && p0 + row < g.pixels && kcol < g.K)
					epi.template load_residual<4>(static_cast<int64_t>(p0 + row) * g.K + kcol, residual[pass]);
			}
		};
		if (VEC && !BY_PIECES) /* (where the pieces take the registers: behind the products, or it waits in scratch memory) */
			request_residual();

		/* LDS rows of 128 bytes, filters behind pixels; chunk c of row r lies in column c ^ (r / 2) % 8: conflict-free to write by rows
		 * and to read by columns.  A wavefront's LDS accesses are done in their order and nobody else touches its part, so the next
		 * stage may be written as soon as the reads of this one are issued: no barrier. */
		const int put = load_row * 8 + (load_chunk ^ (load_row >> 1)); /* rows 8 i + load_row, i even; i odd: column ^ 4 */
		const int r = lane & 31, half = lane >> 5;
		auto walk = [&](auto exact) __attribute__((always_inline))
		{
			for (int s = 0; s < count; s += DEPTH)
			{
#pragma unroll
				for (int d = 0; d < DEPTH; d++)
				{
					/* both operands, so that what lies behind a row (an infinity of the next pixel or tap) counts as nothing */
					uint4 keep = make_uint4(0, 0, 0, 0);
					if (ROW != ROWS_OF_CHUNKS)
						keep = make_uint4(keep_bits(stage[d].left), keep_bits(stage[d].left - 4), keep_bits(stage[d].left - 8), keep_bits(stage[d].left - 12));
#pragma unroll
					for (int q = 0; q < LOADS; q++)
					{
						uint4 xs = stage[d].xs[q].get(origin[q].x + stage[d].x_tap, keep), ws = stage[d].ws[q].get(stage[d].w_at + 8 * q * filter_bytes, keep);
						if constexpr (BY_PIECES && !exact.value)
						{
							xs = scaled(xs);
							ws = scaled(ws);
						}
						mine[64 * q + (q & 1 ? put ^ 4 : put)] = xs;
						mine[8 * SIDE + 64 * q + (q & 1 ? put ^ 4 : put)] = ws;
					}
					wave_order();
					fetch(stage[d]); /* nothing behind the last stage */
					auto plain = [&]() __attribute__((always_inline))
					{
#pragma unroll
						for (int slab = 0; slab < 4; slab++)
						{
							Chunk cw[T], cx[T];
							const int get = r * 8 + ((2 * slab + half) ^ ((r >> 1) & 7));
#pragma unroll
							for (int t = 0; t < T; t++)
							{
								cx[t].u = mine[256 * t + get];
								cw[t].u = mine[8 * SIDE + 256 * t + get];
							}
#pragma unroll
							for (int i = 0; i < T; i++)
#pragma unroll
								for (int j = 0; j < T; j++)
									Mma<TE>::run(cw[i], cx[j], acc[i][j]);
						}
					};
					if constexpr (BY_PIECES)
					{
						if constexpr (exact.value)
							plain();
						else
						{
#pragma unroll
							for (int slab = 0; slab < 4; slab += 2)
							{
								Chunk cw[2][T], cx[2][T];
#pragma unroll
								for (int i = 0; i < 2; i++)
#pragma unroll
									for (int t = 0; t < T; t++)
									{
										const int get = r * 8 + ((2 * (slab + i) + half) ^ ((r >> 1) & 7));
										cx[i][t].u = mine[256 * t + get];
										cw[i][t].u = mine[8 * SIDE + 256 * t + get];
									}
								Pieces pw[T];
#pragma unroll
								for (int i = 0; i < T; i++)
									pw[i].cut(cw[0][i], cw[1][i]);
#pragma unroll
								for (int j = 0; j < T; j++)
								{
									Pieces px;
									px.cut(cx[0][j], cx[1][j]);
#pragma unroll
									for (int n = 0; n < PIECE_PRODUCTS; n++)
#pragma unroll
										for (int i = 0; i < T; i++)
											Mma<bf16_t>::run(pw[i].p[PIECE_OF_A[n]], px.p[PIECE_OF_B[n]], acc[i][j]);
								}
							}
						}
					}
					else
						plain();
					wave_order();
				}
			}
		};
		walk(std::false_type());
		if constexpr (BY_PIECES)
		{
			/* sums that are not finite: this wavefront's share of k once more with fp32 products (struct Pieces) */
			if (__builtin_amdgcn_ballot_w64(!finish_pieces(acc)) != 0)
			{
				begin();
				walk(std::true_type());
			}
			if (VEC)
				request_residual();
		}

		/* a lane holds, of pixel r of each pixel tile, the filters 8 v + 4 (lane / 32) .. + 3 of each filter tile */
		quad_t *part = reinterpret_cast<quad_t*>(mine);
#pragma unroll
		for (int i = 0; i < T; i++)
#pragma unroll
			for (int j = 0; j < T; j++)
#pragma unroll
				for (int v = 0; v < 4; v++)
				{
					quad_t q;
#pragma unroll
					for (int e = 0; e < 4; e++)
						q.v[e] = acc[i][j][4 * v + e];
					part[(8 * i + 2 * v + half) * PITCH + 32 * j + r] = q;
				}
		__syncthreads();
		auto sum_of = [&](int row) __attribute__((always_inline))
		{
			quad_t v = reinterpret_cast<const quad_t*>(lds[0])[quad * PITCH + row];
#pragma unroll
			for (int k = 1; k < KW; k++)
			{
				const quad_t o = reinterpret_cast<const quad_t*>(lds[k])[quad * PITCH + row];
#pragma unroll
				for (int e = 0; e < 4; e++)
					v.v[e] += o.v[e];
			}
			return v;
		};
		auto hand_over = [&](int pass) __attribute__((always_inline))
		{
			const int row = row0 + ROWS * pass;
			if (ROWS > SIDE && row >= SIDE)
				return;
			const quad_t v = sum_of(row);
			if (p0 + row < g.pixels && kcol < g.K)
				epi.template store_at<ACT, VEC, 4>(static_cast<int64_t>(p0 + row) * g.K + kcol, kcol, v.v, columns, VEC ? &residual[VEC ? pass : 0] : nullptr);
		};
		if constexpr (ACT == ACT_VECTORS)
		{
			if (ROWS > SIDE && row0 >= SIDE)
				return;
			float v[PASSES][4];
#pragma unroll
			for (int pass = 0; pass < PASSES; pass++)
			{
				const quad_t q = sum_of(row0 + ROWS * pass);
#pragma unroll
				for (int e = 0; e < 4; e++)
					v[pass][e] = q.v[e];
			}
			epi.store_runs(kcol, v, columns, residual, [&](int pass, int64_t &idx) __attribute__((always_inline))
			{
				const int p = p0 + row0 + ROWS * pass;
				idx = static_cast<int64_t>(p) * g.K + kcol;
				return p < g.pixels && kcol < g.K;
			});
		}
		else if constexpr (ACT == ACT_SIMPLE)
		{
#pragma unroll
			for (int pass = 0; pass < PASSES; pass++)
				hand_over(pass);
		}
		else
		{
#pragma unroll 1 /* the switch over the activations once, not once per pass */
			for (int pass = 0; pass < PASSES; pass++)
				hand_over(pass);
		}
	}
}

namespace
{
	/* only problems of fewer 128 x 128 tiles than this are candidates at all */
	std::atomic<int>& small_problem_threshold()
	{
		static std::atomic<int> value(4096);
		return value;
	}
	/* What the layer takes in them.  `one_tap_us`: the estimate of the persistent one-tap kernels where they take the layer, or 0: what they
	 * decline (filters in no whole runs of 16 bytes) is the gather kernel's and no less than 9 us (bf16 32 -> 20 on 8360 pixels, with a
	 * residual: 11.6 us there, 5.0 in small tiles). */
	double workgroup_tiles_us(const avhipConvShape &s, int element_bytes, HandOver hand_over, double one_tap_us)
	{
		if (hand_over == HandOver::PLAIN && one_tap_us > 0.0)
			return one_tap_us;
		const bool dense = s.stride_h == 1 && s.stride_w == 1 && s.dil_h == 1 && s.dil_w == 1;
		const bool image_tiles = hand_over == HandOver::PLAIN && dense && s.R * s.S > 1 && s.K % 8 == 0 && s.Ho * s.Wo >= 128;
		const int kernel = hand_over == HandOver::PLAIN ? GATHER : hand_over == HandOver::ELEMENTS ? GATHER_BY_ELEMENTS : GATHER_ACTIVATION;
		if (element_bytes == 4 && kernel == GATHER_ACTIVATION && s.K % 4 != 0)
			return tile_kernel_us(s, element_bytes, GATHER_GENERAL);
		if (image_tiles && !(element_bytes == 4 && conv_gather_before_image_tiles(s)))
			return tile_kernel_us(s, element_bytes, IMAGE_TILES);
		return tile_kernel_us(s, element_bytes, kernel);
	}
}

extern "C" int avhip_set_small_problem_threshold(int workgroups)
{
	return small_problem_threshold().exchange(workgroups < 0 ? -1 : workgroups);
}

namespace avhip
{
	int conv_small_threshold()
	{
		return small_problem_threshold().load(std::memory_order_relaxed);
	}
	static bool whole_chunks(const avhipConvShape &s, int element_bytes)
	{
		return static_cast<int64_t>(s.C) * element_bytes % 16 == 0;
	}
	/* taps in a mask; exact division of a chunk's number by multiplication */
	bool conv_small_possible(const avhipConvShape &s, int element_bytes)
	{
		const int64_t chunks = (static_cast<int64_t>(s.C) * element_bytes + 15) / 16;
		return s.R * s.S <= 32 && chunks <= 8192;
	}
	/* The small tiles' estimates are of the plain hand-over; the others cost them up to a fifth of the whole.  Against the one-tap kernels, whose
	 * estimate is the coarsest, they have to be 5 % below. */
	static double small_factor(int element_bytes, HandOver hand_over, double one_tap_us)
	{
		return hand_over != HandOver::PLAIN ? (element_bytes == 4 ? 1.1 : 1.2) : one_tap_us > 0.0 ? 1.05 : 1.0;
	}
	SmallChoice conv_small_choice(const avhipConvShape &s, int element_bytes, HandOver hand_over, double one_tap_us)
	{
		SmallChoice choice = { hand_over, one_tap_us, false, { 0, 0, 0.0, 0.0, 0, 0.0 }, 0.0, false, 0.0 };
		if (!conv_small_possible(s, element_bytes))
			return choice;
		choice.plan = conv_small_plan(s, element_bytes);
		const int threshold = conv_small_threshold();
		if (threshold < 0) /* asked for by name (tests): whatever the kernel can run */
			choice.preferred = choice.larger_preferred = true;
		else if (!whole_chunks(s, element_bytes)) /* otherwise the general gather kernel, element by element: 2.2 to 17 times slower on all of 14 layers of 1152 to 627200 pixels */
			choice.preferred = choice.larger_preferred = threshold != 0;
		else
		{
			choice.us = choice.larger_us = workgroup_tiles_us(s, element_bytes, hand_over, one_tap_us);
			const int64_t tiles = (static_cast<int64_t>(s.N) * s.Ho * s.Wo + 127) / 128 * ((static_cast<int64_t>(s.K) + 127) / 128);
			const double limit = tiles < threshold ? choice.us / small_factor(element_bytes, hand_over, one_tap_us) : 0.0;
			choice.larger_preferred = choice.plan.larger_us > 0.0 && choice.plan.larger_us < limit;
			/* (tiles of 16 x 16 against the one-tap kernels in 16 and 8 bits: those take 4.0 to 4.3 us for one stage where they are estimated at 5.2, for two 4.7 to 5.2; so 13 % below for one.  With 5 % layers of 3600 to 4900
			 * such tiles were slower, int8 80 -> 80 on 15652 pixels 4.1 -> 5.0 us, bf16 64 -> 64 on 16632 4.2 -> 4.6) */
			const bool loose = choice.plan.side == 16 && element_bytes < 4 && one_tap_us > 0.0 && static_cast<int64_t>(s.C) * element_bytes <= 128;
			choice.preferred = choice.plan.us < (loose ? 0.92 * limit : limit) || (choice.plan.side == 16 && choice.larger_preferred);
		}
		const double factor = small_factor(element_bytes, hand_over, 0.0);
		if (choice.preferred)
			choice.us = factor * choice.plan.us;
		if (choice.larger_preferred)
			choice.larger_us = factor * choice.plan.larger_us;
		return choice;
	}
	bool conv_gather_before_image_tiles(const avhipConvShape &s)
	{
		return tile_kernel_us(s, 4, GATHER) < tile_kernel_us(s, 4, IMAGE_TILES);
	}

	template<typename TE, typename Epi>
	bool conv_small_launch(hipStream_t stream, const avhipConvShape &s, const void *x, const void *w, const Epi &epi, const SmallChoice &choice)
	{
		constexpr int SZ = static_cast<int>(sizeof(TE));
		const int64_t pixels = static_cast<int64_t>(s.N) * s.Ho * s.Wo;
		const SmallPlan &plan = choice.plan;
		const bool simple = choice.hand_over == HandOver::PLAIN;
		if (!choice.preferred || in_place(s, x, SZ, epi.y, Epi::out_bytes))
			return false;
		const int side = plan.side;
		const int64_t pixel_tiles = (pixels + side - 1) / side, filter_tiles = (static_cast<int64_t>(s.K) + side - 1) / side;
		if (pixel_tiles * 64 * plan.waves >= (1ll << 32) /* work-items of a launch along one direction */ || filter_tiles > 65535
				|| pixel_tiles * filter_tiles > 0x7FFFFFFFll || pixels >= (1ll << 31) - side)
			return false;
		const SmallGeom g = small_geometry(s, SZ, pixel_tiles, filter_tiles);
		const dim3 grid(g.pixel_tiles, g.filter_tiles);
		if (side == 16)
		{
			conv_small16_launch<TE, Epi>(stream, grid, plan.waves, x, w, g, epi, choice.hand_over);
			return true;
		}
		/* All results of a work-item at once, with the residual requested ahead, where that is the faster way: for rows of dwords in tiles of 32 x 32 the registers of it (132 to 148 a lane, 128 without)
		 * cost one wavefront in four of a SIMD, which ELU and SELU repay (1.04 to 1.19 times as fast) and the library's functions do not (16 layers 0.985 on average, f16 66 -> 64 1x1 stride 2 with
		 * tanh on 256 x 28 x 29 12.4 -> 13.8 us). */
		const bool dword_rows = !whole_chunks(s, SZ) && (s.C * SZ) % 4 == 0;
		const bool runs = Epi::runs && epi.vec && choice.hand_over == HandOver::ACTIVATION
				&& !(side == 32 && dword_rows && epi.activation != ACT_ELU && epi.activation != ACT_SELU);
#define AVHIP_SMALL_PLAN(T, KW, ROW) \
		do \
		{ \
			if (simple) \
				hipLaunchKernelGGL((k_conv_small<TE, Epi, T, KW, ACT_SIMPLE, ROW>), grid, dim3(64 * KW), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi); \
			else if (runs) \
				hipLaunchKernelGGL((k_conv_small<TE, Epi, T, KW, Epi::runs ? ACT_VECTORS : ACT_ANY, ROW>), grid, dim3(64 * KW), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi); \
			else \
				hipLaunchKernelGGL((k_conv_small<TE, Epi, T, KW, ACT_ANY, ROW>), grid, dim3(64 * KW), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi); \
		} while (0)
#define AVHIP_SMALL(ROW) \
		do \
		{ \
			if (side == 64) \
				AVHIP_SMALL_PLAN(2, 4, ROW); \
			else if (plan.waves == 8) \
				AVHIP_SMALL_PLAN(1, 8, ROW); \
			else if (plan.waves == 4) \
				AVHIP_SMALL_PLAN(1, 4, ROW); \
			else \
				AVHIP_SMALL_PLAN(1, 1, ROW); \
		} while (0)
		if (!whole_chunks(s, SZ))
		{
			if (SZ == 4 || (SZ == 2 && s.C % 2 == 0))
			{
				if constexpr (SZ >= 2)
					AVHIP_SMALL(ROWS_OF_DWORDS);
			}
			else if constexpr (SZ <= 2)
				AVHIP_SMALL(ROWS_OF_ELEMENTS);
		}
		else
			AVHIP_SMALL(ROWS_OF_CHUNKS);
#undef AVHIP_SMALL
#undef AVHIP_SMALL_PLAN
		return true;
	}

#define AVHIP_INSTANTIATE(TE, EPI) template bool conv_small_launch<TE, EPI>(hipStream_t, const avhipConvShape&, const void*, const void*, const EPI&, const SmallChoice&);
	AVHIP_INSTANTIATE(float, FloatEpilogue<float>)
	AVHIP_INSTANTIATE(f16_t, FloatEpilogue<f16_t>)
	AVHIP_INSTANTIATE(bf16_t, FloatEpilogue<bf16_t>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_EXACT>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_REQUANT>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_FLOAT_I32>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_FLOAT_I8>)
	AVHIP_INSTANTIATE(int8_t, Int8Epilogue<I8_FLOAT_F32>)
#undef AVHIP_INSTANTIATE
}

/* The tile that a layer of more than one tap (of fp32, or one that the ring kernel leaves alone) gets in this kernel: half of its side
 * plus wavefronts, or 0 where it goes to another.  `hand_over`: HandOver.  Exported so that a test can ask which instance it is about to run. */
extern "C" AVHIP_API int avhip_conv2d_small_plan(int x_dtype, const avhipConvShape *shape, int hand_over)
{
	if (shape == nullptr || hand_over < 0 || hand_over > 2)
		return 0;
	const int element_bytes = x_dtype == DT_INT8 ? 1 : x_dtype == DT_FLOAT32 ? 4 : 2;
	const SmallChoice choice = conv_small_choice(*shape, element_bytes, static_cast<HandOver>(hand_over), 0.0);
	return choice.preferred ? choice.plan.side / 2 + choice.plan.waves : 0;
}

extern "C" AVHIP_API double avhip_conv2d_small_us(int x_dtype, const avhipConvShape *shape, int hand_over)
{
	if (shape == nullptr || hand_over < 0 || hand_over > 2 || conv_small_threshold() <= 0)
		return 0.0;
	const int element_bytes = x_dtype == DT_INT8 ? 1 : x_dtype == DT_FLOAT32 ? 4 : 2;
	return whole_chunks(*shape, element_bytes) ? conv_small_choice(*shape, element_bytes, static_cast<HandOver>(hand_over), 0.0).us : 0.0;
}

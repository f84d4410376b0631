/*
 * conv_small16.hip -- implicit-GEMM convolution in tiles of 16 x 16, for layers whose tiles of 32 x 32 leave most of the chip idle.
 *
 * As k_conv_small (conv_small.hip): k is shared by the one, four or eight wavefronts of a workgroup, each brings its operands by rows of 128 bytes through LDS of its own into the MFMA's
 * layout, the partial tiles are added through LDS in a fixed order.  What bound that kernel on the smallest layers, by the clock inside it (fp16 128 -> 128 3x3 on one image of 15 x 15, 32 tiles,
 * 6.3 us): 0.6 us until a pixel's address and border mask were known, then 3.0 us in which a compute unit loaded 147 KB at its 64 bytes a clock (1.05 us at least) in two
 * stages at a time, 0.7 us for sums and results, 1.7 us of launch.  So: tiles of a quarter, for four times as many compute units (half as many bytes each; in fp32 a quarter of the products);
 * the filters' loads before the pixels' addresses; the border by two comparisons a load and not by a mask made in loops.  One pixel quad a lane is left to hand over: the first wavefront does.
 * What bounds it now: the latency of one load, the sums and the launch, 2.8 us of them for a layer of one stage.
 * Measured, before (tiles of 32 x 32) and now: that layer 5.9 -> 4.1 us, bf16 256 -> 256 3x3 on 3 x 13 x 13 7.8 -> 6.7, fp32 64 -> 64 3x3 on 8 x 15 x 15 8.2 -> 5.6, fp32 128 -> 128 on
 * 512 pixels 11.3 -> 5.6, int8 1x1 48 -> 48 on 320 pixels 3.6 -> 2.7; 1584 16-bit layers that the estimates send here are 1.26 times as fast, 298 of fp32 1.48 times.
 * Rows of dwords and elements (any number of channels) against tiles of 32 x 32: bf16 97 -> 32 3x3 stride 2 on 364 pixels 6.7 -> 4.4 us, fp32 133 -> 32 3x3 on 640 11.6 -> 6.4; few channels against
 * the kernels made for them: fp32 4 -> 128 3x3 on 6 x 11 x 11 8.8 -> 3.3, fp16 8 -> 80 3x3 on 845 pixels 6.0 -> 3.2, bf16 4 -> 128 on 512 4.4 -> 3.4.
 * Three or four stages in flight and sixteen wavefronts were not faster, two wavefronts in no layer by more than 5 %.
 */
#include "conv_small.hpp"
#include "conv_small_rows.hpp"
#include "mfma_core.hpp"

namespace
{
	using namespace avhip;

	typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

	/* One 16 x 16 accumulator tile: a lane holds rows 4 (lane / 16) .. + 3 of column lane % 16, and of a chunk pair row lane % 16, chunk lane / 16 of four. */
	template<typename TE> struct Mma16;
	template<> struct Mma16<bf16_t>
	{
		typedef f32x4_t acc_t;
		__device__ static __forceinline__ void run(const Chunk &a, const Chunk &b, acc_t &c)
		{
			c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.bf, b.bf, c, 0, 0, 0);
		}
	};
	template<> struct Mma16<f16_t>
	{
		typedef f32x4_t acc_t;
		__device__ static __forceinline__ void run(const Chunk &a, const Chunk &b, acc_t &c)
		{
			c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.hf, b.hf, c, 0, 0, 0);
		}
	};
	template<> struct Mma16<int8_t>
	{
		typedef i32x4_t acc_t;
		__device__ static __forceinline__ void run(const Chunk &a, const Chunk &b, acc_t &c)
		{
			c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a.i4, b.i4, c, 0, 0, 0);
		}
	};
	template<> struct Mma16<float>
	{
		typedef f32x4_t acc_t;
		__device__ static __forceinline__ void run(const Chunk &a, const Chunk &b, acc_t &c)
		{
#pragma unroll
			for (int i = 0; i < 4; i++)
				c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.f[i], b.f[i], c, 0, 0, 0);
		}
	};

	/* KW wavefronts on one tile */
	template<typename TE, typename Epi, int KW, int ACT, int ROW>
	__global__ __launch_bounds__(64 * KW, 4) void k_conv_small16(const TE *__restrict__ x, const TE *__restrict__ w, SmallGeom g, Epi epi)
	{
		constexpr unsigned int SZ = sizeof(TE);
		constexpr int SIDE = 16;
		constexpr int DEPTH = 2; /* stages of a wavefront in flight; of more, short shares pay for loads of nothing */
		constexpr bool VEC = ACT != ACT_ANY;
		typedef typename Epi::scalar_t scalar_t;
		typedef Pack<scalar_t, 4> quad_t;
		/* each wavefront its own part: 16 rows of 128 bytes of either operand, then its partial tile */
		__shared__ __attribute__((aligned(16))) uint4 lds[KW][2 * SIDE * 8];

		const int lane = threadIdx.x & 63;
		const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
		uint4 *mine = lds[wave];
		/* the order of the tiles: as k_conv_small */
		const unsigned int t = xcd_block(blockIdx.y * g.pixel_tiles + blockIdx.x, g.pixel_tiles * g.filter_tiles);
		const unsigned int slow = g.by_tiles.of(t), fast = t - slow * (g.pixels_first ? g.pixel_tiles : g.filter_tiles);
		const unsigned int pixel_tile = g.pixels_first ? fast : slow, filter_tile = g.pixels_first ? slow : fast;
		const int p0 = static_cast<int>(pixel_tile) * SIDE, k0 = static_cast<int>(filter_tile) * SIDE;

		const unsigned int c_bytes = g.C * SZ, filter_bytes = g.R * g.S * c_bytes;
		const __amdgpu_buffer_rsrc_t rx = make_buffer(x, (static_cast<unsigned int>(g.images) * g.H * g.W * c_bytes + 3) & ~3u); /* a dword never crosses a page */
		const __amdgpu_buffer_rsrc_t rw = make_buffer(w, (static_cast<unsigned int>(g.K) * filter_bytes + 3) & ~3u);

		/* k = the 16-byte chunks of (tap, channel) in a row, eight a stage; each wavefront takes a contiguous share of the stages.  This lane loads chunk
		 * (lane % 8) of the rows 8 i + lane / 8. */
		const int load_row = lane >> 3, load_chunk = lane & 7;
		const unsigned int w_origin = static_cast<unsigned int>(k0 + load_row) * filter_bytes; /* filters past the last lie outside the buffer */
		const int chunks = g.R * g.S * g.chunks_per_tap;
		const int stages = (chunks + 7) / 8;
		const int share = (stages + KW - 1) / KW;
		const int first = wave * share;
		const int count = stages - first < share ? stages - first : share; /* may be negative: nothing left for this wavefront */
		const unsigned int chunks_mine = count > 0 ? (chunks < 8 * (first + count) ? chunks : 8 * (first + count)) : 0;
		struct Stage
		{
			Piece<ROW> xs[2], ws[2];
			unsigned int x_tap, w_at; /* not whole chunks: where the pieces start (the lowest two bits are used) */
			int left; /* and the bytes of the row from there */
		};
		Stage stage[DEPTH];
		unsigned int w_chunk = 8 * first + load_chunk, x_chunk = w_chunk;
		auto tap_of = [&](unsigned int chunk) __attribute__((always_inline))
		{
			return g.chunks_per_tap == 1 ? chunk : __umulhi(chunk, g.by_chunks); /* (one chunk a tap: the factor would be 2^32) */
		};
		auto fetch_w = [&](Stage &to) __attribute__((always_inline))
		{
			unsigned int at = w_origin + 16 * w_chunk;
			if (ROW != ROWS_OF_CHUNKS)
			{
				const unsigned int tap = tap_of(w_chunk), c = w_chunk - tap * g.chunks_per_tap;
				at = w_origin + tap * c_bytes + 16 * c;
				to.w_at = at;
				to.left = static_cast<int>(c_bytes - 16 * c);
			}
#pragma unroll
			for (int q = 0; q < 2; q++)
				to.ws[q].fetch(rw, w_chunk < chunks_mine ? at + 8 * q * filter_bytes : OUT_OF_RANGE);
			w_chunk += 8;
		};
		/* the filters' operands are on their way while the pixels' addresses are worked out */
#pragma unroll
		for (int d = 0; d < DEPTH; d++)
			fetch_w(stage[d]);
		int ih0[2], iw0[2];
		unsigned int origin[2];
#pragma unroll
		for (int q = 0; q < 2; q++)
		{
			const int p = p0 + 8 * q + load_row;
			const int pp = p < g.pixels ? p : 0;
			const int line = static_cast<int>(g.by_wo.of(pp)), ow = pp - line * g.Wo;
			const int n = static_cast<int>(g.by_ho.of(line)), oh = line - n * g.Ho;
			ih0[q] = oh * g.stride_h + g.pad_h;
			iw0[q] = ow * g.stride_w + g.pad_w;
			origin[q] = static_cast<unsigned int>((n * g.H + ih0[q]) * g.W + iw0[q]) * c_bytes;
			if (p >= g.pixels)
				ih0[q] = -(1 << 30); /* no tap of it lies inside */
		}
		auto fetch_x = [&](Stage &to) __attribute__((always_inline))
		{
			const unsigned int tap = tap_of(x_chunk), c = x_chunk - tap * g.chunks_per_tap;
			const unsigned int ti = (tap * g.by_s) >> 16, tj = tap - ti * g.S;
			const int i = static_cast<int>(g.flip ? g.R - 1 - ti : ti) * g.dil_h, j = static_cast<int>(g.flip ? g.S - 1 - tj : tj) * g.dil_w;
			const unsigned int x_tap = static_cast<unsigned int>(i * g.W + j) * c_bytes + 16 * c;
			if (ROW != ROWS_OF_CHUNKS)
				to.x_tap = x_tap;
#pragma unroll
			for (int q = 0; q < 2; q++)
			{
				const bool inside = x_chunk < chunks_mine && static_cast<unsigned int>(ih0[q] + i) < static_cast<unsigned int>(g.H)
						&& static_cast<unsigned int>(iw0[q] + j) < static_cast<unsigned int>(g.W);
				to.xs[q].fetch(rx, inside ? origin[q] + x_tap : OUT_OF_RANGE);
			}
			x_chunk += 8;
		};
#pragma unroll
		for (int d = 0; d < DEPTH; d++)
			fetch_x(stage[d]);

		/* what the epilogue, the first wavefront's, needs is requested behind the first operands: four lanes have a pixel */
		const int quad = lane & 3, row = lane >> 2, kcol = k0 + 4 * quad;
		const bool exists = p0 + row < g.pixels && kcol < g.K;
		const int64_t idx = static_cast<int64_t>(p0 + row) * g.K + kcol;
		typename Epi::Columns columns;
		typename Epi::template Residual<4> residual[1];
		if (wave == 0)
		{
			epi.load_columns(kcol, columns);
			if (VEC && exists)
				epi.template load_residual<4>(idx, residual[0]);
		}

		/* LDS rows of 128 bytes, filters behind pixels; chunk c of row r lies in column c ^ (r / 2) % 8: conflict-free to write by rows and to read by
		 * columns.  A wavefront's LDS accesses are done in their order: no barrier. */
		const int put = load_row * 8 + (load_chunk ^ (load_row >> 1)); /* row 8 + load_row: column ^ 4 */
		const int r = lane & 15, part = lane >> 4;
		typename Mma16<TE>::acc_t acc = { 0, 0, 0, 0 };
		auto bring = [&](const Stage &from) __attribute__((always_inline))
		{
			/* both operands, so that what lies behind a row (an infinity of the next pixel or tap) counts as nothing */
			uint4 keep = make_uint4(0, 0, 0, 0);
			if (ROW != ROWS_OF_CHUNKS)
				keep = make_uint4(keep_bits(from.left), keep_bits(from.left - 4), keep_bits(from.left - 8), keep_bits(from.left - 12));
#pragma unroll
			for (int q = 0; q < 2; q++)
			{
				mine[64 * q + (q ? put ^ 4 : put)] = from.xs[q].get(origin[q] + from.x_tap, keep);
				mine[8 * SIDE + 64 * q + (q ? put ^ 4 : put)] = from.ws[q].get(from.w_at + 8 * q * filter_bytes, keep);
			}
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		};
		auto multiply = [&]() __attribute__((always_inline))
		{
			Chunk cx[2], cw[2];
#pragma unroll
			for (int slab = 0; slab < 2; slab++)
			{
				const int get = r * 8 + ((4 * slab + part) ^ (r >> 1));
				cx[slab].u = mine[get];
				cw[slab].u = mine[8 * SIDE + get];
			}
#pragma unroll
			for (int slab = 0; slab < 2; slab++)
				Mma16<TE>::run(cw[slab], cx[slab], acc);
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		};
		int left = count;
		for (; left > DEPTH; left -= DEPTH)
		{
#pragma unroll
			for (int d = 0; d < DEPTH; d++)
			{
				bring(stage[d]);
				fetch_w(stage[d]); /* nothing behind the last stage */
				fetch_x(stage[d]);
				multiply();
			}
		}
#pragma unroll
		for (int d = 0; d < DEPTH; d++)
			if (d < left)
			{
				bring(stage[d]);
				multiply();
			}

		/* a lane holds the filters 4 part .. + 3 of pixel r; the partial tiles are added in a fixed order */
		quad_t q;
#pragma unroll
		for (int e = 0; e < 4; e++)
			q.v[e] = acc[e];
		reinterpret_cast<quad_t*>(mine)[part * SIDE + r] = q;
		__syncthreads();
		if (wave != 0)
			return;
		quad_t v = reinterpret_cast<const quad_t*>(lds[0])[quad * SIDE + row];
#pragma unroll
		for (int k = 1; k < KW; k++)
		{
			const quad_t o = reinterpret_cast<const quad_t*>(lds[k])[quad * SIDE + row];
#pragma unroll
			for (int e = 0; e < 4; e++)
				v.v[e] += o.v[e];
		}
		if constexpr (ACT == ACT_VECTORS)
		{
			float run[1][4];
#pragma unroll
			for (int e = 0; e < 4; e++)
				run[0][e] = v.v[e];
			epi.store_runs(kcol, run, columns, residual, [&](int, int64_t &at) __attribute__((always_inline))
			{
				at = idx;
				return exists;
			});
		}
		else if (exists)
			epi.template store_at<ACT, VEC, 4>(idx, kcol, v.v, columns, VEC ? &residual[0] : nullptr);
	}
}

namespace avhip
{
	template<typename TE, typename Epi>
	void conv_small16_launch(hipStream_t stream, const dim3 &grid, int waves, const void *x, const void *w, const SmallGeom &g, const Epi &epi, HandOver hand_over)
	{
#define AVHIP_SMALL16_ACT(KW, ROW, ACT) hipLaunchKernelGGL((k_conv_small16<TE, Epi, KW, ACT, ROW>), grid, dim3(64 * KW), 0, stream, static_cast<const TE*>(x), static_cast<const TE*>(w), g, epi)
#define AVHIP_SMALL16_WAVES(KW, ROW) \
		do \
		{ \
			if (hand_over == HandOver::PLAIN) \
				AVHIP_SMALL16_ACT(KW, ROW, ACT_SIMPLE); \
			else if (Epi::runs && epi.vec && hand_over == HandOver::ACTIVATION) \
				AVHIP_SMALL16_ACT(KW, ROW, Epi::runs ? ACT_VECTORS : ACT_ANY); \
			else \
				AVHIP_SMALL16_ACT(KW, ROW, ACT_ANY); \
		} while (0)
#define AVHIP_SMALL16(ROW) \
		do \
		{ \
			if (waves == 8) \
				AVHIP_SMALL16_WAVES(8, ROW); \
			else if (waves == 4) \
				AVHIP_SMALL16_WAVES(4, ROW); \
			else \
				AVHIP_SMALL16_WAVES(1, ROW); \
		} while (0)
		constexpr int SZ = static_cast<int>(sizeof(TE));
		if (g.C * SZ % 16 == 0)
			AVHIP_SMALL16(ROWS_OF_CHUNKS);
		else if (g.C * SZ % 4 == 0)
		{
			if constexpr (SZ >= 2)
				AVHIP_SMALL16(ROWS_OF_DWORDS);
			else
				AVHIP_SMALL16(ROWS_OF_ELEMENTS);
		}
		else if constexpr (SZ <= 2)
			AVHIP_SMALL16(ROWS_OF_ELEMENTS);
#undef AVHIP_SMALL16
#undef AVHIP_SMALL16_WAVES
#undef AVHIP_SMALL16_ACT
	}

#define AVHIP_INSTANTIATE(TE, EPI) template void conv_small16_launch<TE, EPI>(hipStream_t, const dim3&, int, const void*, const void*, const SmallGeom&, const EPI&, HandOver);
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

/*
 * conv_winograd_f4.hip -- y = act(alpha1 * conv(x, w) + bias + alpha2 * z) + beta * y in fp32 by Winograd F(4x4, 3x3) in ONE kernel.
 *
 * The mathematics of the non-fused plan (src/winograd_nonfused.cu:257-519 of the reference, tables 534-575) without its matrices V and
 * M in memory: for 256 images of 15 x 15 with 128 channels these are 75 MB each, written and read once, and that traffic and not the
 * 4.8 GFLOP of the products was what bounded the plan (16 + 56 + 18 us).
 *
 *   workgroup = 32 tiles (of 4 x 4 output pixels, in the order of the images) x 64 filters, eight wavefronts: four groups of nine
 *               transform points x two halves of the filters; a wavefront keeps its nine 32 x 32 products in 144 registers over the
 *               whole of k.  4096 tiles x 128 filters are 256 workgroups, one per compute unit;
 *   input     : per stage of 16 channels a work-item loads the 6 x 6 pixels of one tile and channel, transforms them in registers and
 *               writes 36 dwords of V to LDS (two buffers of 72 KB, one barrier a stage).  Wavefronts 0 to 3 do this before their
 *               products and 4 to 7 behind them: one of each kind shares a SIMD, so the vector ALU works under the other's MFMAs;
 *   weights   : U in operand order (avhip_winograd_f4_weight_transform), one contiguous kilobyte per load, six loads ahead;
 *   output    : M through LDS, 32 filters at a time, A^T M A in registers, the shared epilogue.
 *
 * What bounds it: the matrix cores during the stages (3.8 us for 36 x 32 x 64 x 16 products at 256 flop a clock, 4.8 measured), and
 * around them some 20 us in which all compute units load their first tiles and write their results.  How much of those is the HBM's is not
 * known: every instance has 256 vector registers and spills (272 bytes of scratch a work-item, 292 with a residual: 36 to 38 MB a launch of
 * 256 workgroups, where x and y are 29.5), in front of the first loop, a few in every stage and in both passes of the output.
 * Measured, three passes before and now, one layer again and again from a graph: 256 x 15 x 15 x 128 -> 128 87 -> 61 us, with a residual 91 ->
 * 70 us (a tower of 20 of them in turn, 1925 -> 1422 us, is 68 and 75 us a layer), 64 channels 49 -> 36 us, 40 x 40 x 40 x 99 -> 128 118 -> 60 us,
 * 32 x 56 x 56 x 64 -> 64 with residual 77 -> 47 us, 60 x 28 x 28 x 128 -> 128 68 -> 59 us.  Relative error against 64 bits 1.2e-6 to 2.9e-6 as
 * before (each within 3 % below).
 */
#include <type_traits>

#include "conv_epilogue.hpp"
#include "conv_winograd_f4.hpp"
#include "mfma_core.hpp"

namespace
{
	using namespace avhip;

	constexpr int POINTS = 36;
	constexpr int TILES = 32; /* of a workgroup */
	constexpr int FILTERS = 64;
	constexpr int CHANNELS = 16; /* of a stage */
	constexpr int MY_POINTS = 9; /* of a wavefront */
	constexpr int STEPS = MY_POINTS * CHANNELS / 8; /* loads of U per wavefront and stage */
	constexpr int AHEAD = 6; /* of them in flight */
	static_assert(STEPS % AHEAD == 0, "the slots of the loads in flight are the same in every stage");

	struct F4Geom
	{
		int H, W, C, K, tiles, tiles_h, tiles_w, pad_h, pad_w;
		unsigned int x_bytes, u_bytes, y_bytes;
		int stages, filter_blocks;
	};

	/* offsets beyond every tensor the launcher accepts (below 2^29 bytes), alone and added up */
	constexpr unsigned int NO_ROW = 0x80000000u, NO_COLUMN = 0x40000000u, NO_CHANNEL = 0x20000000u;

	/* B^T d along one direction: [1 0 -5/4 0 1/4 0; 0 1 1 -1/4 -1/4 0; 0 -1 1 1/4 -1/4 0; 0 -1 -1/2 1 1/2 0; 0 1 -1/2 -1 1/2 0; 0 1 0 -5/4 0 1/4] */
	__device__ __forceinline__ void input_line(float &d0, float &d1, float &d2, float &d3, float &d4, float &d5)
	{
		const float a = d2 - 0.25f * d4, b = d1 - 0.25f * d3, c = d4 - d2, e = d3 - d1;
		const float o0 = (d0 + 0.25f * c) - d2, o5 = 0.25f * (d5 - d3) - e;
		d0 = o0;
		d1 = a + b;
		d2 = a - b;
		d3 = e + 0.5f * c;
		d4 = 0.5f * c - e;
		d5 = o5;
	}
	/* A^T m along one direction: [1 1 1 1/4 1/4 0; 0 1 -1 1/2 -1/2 0; 0 1 1 1 1 0; 0 1 -1 2 -2 2] */
	__device__ __forceinline__ void output_line(const float (&m)[6], float (&y)[4])
	{
		const float s = m[1] + m[2], t = m[1] - m[2], u = m[3] + m[4], v = m[3] - m[4];
		y[0] = m[0] + s + 0.25f * u;
		y[1] = t + 0.5f * v;
		y[2] = s + u;
		y[3] = t + 2.0f * (v + m[5]);
	}

	template<bool RELU, bool RESIDUAL>
	__global__ __launch_bounds__(512, 2) void k_winograd_f4(const float *__restrict__ x, const float *__restrict__ U, F4Geom g, FloatEpilogue<float> epi)
	{
		/* V: [point][quad of channels][tile][channel of the quad]; M: [point][quad of filters][tile][filter of the quad], tiles in
		 * the order tile ^ 4 * quad: conflict-free for the work-items of neighbouring quads and for those of neighbouring tiles */
		constexpr int V_FLOATS = POINTS * CHANNELS * TILES;
		static_assert(2 * V_FLOATS == POINTS * 32 * TILES, "the products of half of the filters take the place of the two stages");
		__shared__ __attribute__((aligned(16))) float lds[2 * V_FLOATS];

		const int tid = threadIdx.x, lane = tid & 63;
		const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
		const int first_point = MY_POINTS * (wave & 3), my_half = wave >> 2;
		/* the filter blocks of a tile block are neighbours: their input comes from one L2 */
		const unsigned int block = xcd_block(blockIdx.x, gridDim.x);
		const unsigned int tile_block = block / g.filter_blocks, filter_block = block - tile_block * g.filter_blocks;
		const int t0 = static_cast<int>(tile_block) * TILES, k0 = static_cast<int>(filter_block) * FILTERS;

		const __amdgpu_buffer_rsrc_t rx = make_buffer(x, g.x_bytes);
		const __amdgpu_buffer_rsrc_t ru = make_buffer(U, g.u_bytes);
		const __amdgpu_buffer_rsrc_t ry = make_buffer(epi.y, g.y_bytes), rz = make_buffer(RESIDUAL ? epi.z : epi.y, g.y_bytes);

		/* one tile and one channel of a stage per work-item */
		const int tile = tid >> 4, channel = tid & 15;
		const int t = t0 + tile;
		const int line = t / g.tiles_w, tw = t - line * g.tiles_w;
		const int image = line / g.tiles_h, th = line - image * g.tiles_h;
		unsigned int row[6], column[6];
#pragma unroll
		for (int a = 0; a < 6; a++)
		{
			const int ih = 4 * th + g.pad_h + a, iw = 4 * tw + g.pad_w + a;
			row[a] = t < g.tiles && ih >= 0 && ih < g.H
					? static_cast<unsigned int>(((image * g.H + ih) * g.W + 4 * tw + g.pad_w) * g.C + channel) * 4u : NO_ROW;
			column[a] = iw >= 0 && iw < g.W ? static_cast<unsigned int>(a * g.C) * 4u : NO_COLUMN;
		}
		float d[36];
		auto load_input = [&](int stage) __attribute__((always_inline))
		{
			const unsigned int at = 64u * stage + (CHANNELS * stage + channel < g.C ? 0u : NO_CHANNEL);
#pragma unroll
			for (int a = 0; a < 6; a++)
			{
				unsigned int line = row[a] + at;
				asm volatile("" : "+v"(line)); /* or 36 sums of row and column are kept over the loop, more than there are registers */
#pragma unroll
				for (int b = 0; b < 6; b++)
					d[6 * a + b] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, static_cast<int>(line + column[b]), 0, 0));
				__builtin_amdgcn_sched_barrier(0); /* six offsets at a time */
			}
		};
		const int put = (channel >> 2) * (TILES * 4) + (tile ^ (channel & ~3)) * 4 + (channel & 3);
		auto transform_input = [&](int buffer) __attribute__((always_inline))
		{
			float *to = lds + buffer * V_FLOATS + put;
#pragma unroll
			for (int b = 0; b < 6; b++)
				input_line(d[b], d[6 + b], d[12 + b], d[18 + b], d[24 + b], d[30 + b]);
#pragma unroll
			for (int a = 0; a < 6; a++)
			{
				input_line(d[6 * a], d[6 * a + 1], d[6 * a + 2], d[6 * a + 3], d[6 * a + 4], d[6 * a + 5]);
#pragma unroll
				for (int b = 0; b < 6; b++)
					to[(6 * a + b) * (CHANNELS * TILES)] = d[6 * a + b];
			}
		};

		/* U: [block of 32 filters][point][8 channels][lane][4 channels]; step i of a stage: point i / 2, half i % 2 of its channels */
		const int slabs = 2 * g.stages;
		const int u_first = ((2 * static_cast<int>(filter_block) + my_half) * POINTS + first_point) * slabs;
		uint4 u[AHEAD];
		auto load_weights = [&](int step, int stage) __attribute__((always_inline))
		{
			const int slab = u_first + (step >> 1) * slabs + 2 * stage + (step & 1);
			u[step % AHEAD] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ru, lane * 16, slab * 1024, 0));
		};
		Mma<float>::acc_t acc[MY_POINTS]; /* [filters][tiles] */
#pragma unroll
		for (int p = 0; p < MY_POINTS; p++)
#pragma unroll
			for (int v = 0; v < 16; v++)
				acc[p][v] = 0;
		const int r = lane & 31, half = lane >> 5;
		auto multiply = [&](int stage, int next) __attribute__((always_inline))
		{
			const uint4 *from = reinterpret_cast<const uint4*>(lds + (stage & 1) * V_FLOATS) + first_point * (CHANNELS / 4 * TILES);
			Chunk cx[2];
			auto read = [&](int i) __attribute__((always_inline))
			{
				const int quad = 2 * (i & 1) + half;
				cx[i & 1].u = from[((i >> 1) * (CHANNELS / 4) + quad) * TILES + (r ^ (4 * quad))];
			};
			read(0);
#pragma unroll
			for (int i = 0; i < STEPS; i++)
			{
				if (i + 1 < STEPS)
					read(i + 1);
				Chunk cw;
				cw.u = u[i % AHEAD];
				Mma<float>::run(cw, cx[i & 1], acc[i >> 1]);
				if (i + AHEAD < STEPS)
					load_weights(i + AHEAD, stage);
				else
					load_weights(i + AHEAD - STEPS, next);
				/* without it the loads are moved down to their use and every step waits for its own */
				__builtin_amdgcn_sched_barrier(0);
			}
		};

		load_input(0);
#pragma unroll
		for (int i = 0; i < AHEAD; i++)
			load_weights(i, 0);
		transform_input(0);
		load_input(1); /* (behind the last channel: zeros) */
		const int last = g.stages - 1;
		if (wave < 4)
			for (int s = 0; s < last; s++)
			{
				__syncthreads(); /* V of this stage is complete, that of the one before has been read */
				transform_input((s + 1) & 1);
				load_input(s + 2);
				multiply(s, s + 1);
			}
		else
			for (int s = 0; s < last; s++)
			{
				__syncthreads();
				multiply(s, s + 1);
				transform_input((s + 1) & 1);
				load_input(s + 2);
			}
		__syncthreads();
		multiply(last, last); /* (the loads ahead: its own weights once more) */

		/* two filters of a tile per work-item: its place among 16 neighbours is the pair, so that runs of 128 bytes leave */
		const int pair = tid & 15;
		float4 *products = reinterpret_cast<float4*>(lds);
#pragma unroll
		for (int pass = 0; pass < 2; pass++)
		{
			const int k = k0 + 32 * pass + 2 * pair;
			FloatEpilogue<float>::ColumnsT<2> columns;
			epi.load_columns(k, columns);
			const int oh0 = 4 * th, ow0 = 4 * tw;
			const bool exists = t < g.tiles && k < g.K;
			const unsigned int first = static_cast<unsigned int>(((image * g.H + oh0) * g.W + ow0) * g.K + k) * 4u;
			auto place = [&](int a, int b) __attribute__((always_inline))
			{
				return exists && oh0 + a < g.H && ow0 + b < g.W ? first + static_cast<unsigned int>((a * g.W + b) * g.K) * 4u : OUT_OF_RANGE;
			};
			typedef float pair_t __attribute__((ext_vector_type(2)));
			pair_t residual[2][4]; /* of a column of pixels, the next one's behind it */
			auto load_residual = [&](int b) __attribute__((always_inline))
			{
#pragma unroll
				for (int a = 0; a < 4; a++)
					residual[b & 1][a] = __builtin_bit_cast(pair_t, __builtin_amdgcn_raw_buffer_load_b64(rz, static_cast<int>(place(a, b)), 0, 0));
			};
			if (RESIDUAL)
				load_residual(0);
			__syncthreads();
			if (my_half == pass)
			{
#pragma unroll
				for (int p = 0; p < MY_POINTS; p++)
#pragma unroll
					for (int v = 0; v < 4; v++)
					{
						const int quad = 2 * v + half;
						products[((first_point + p) * 8 + quad) * TILES + (r ^ (4 * quad))] = make_float4(acc[p][4 * v], acc[p][4 * v + 1], acc[p][4 * v + 2], acc[p][4 * v + 3]);
					}
			}
			__syncthreads();
			const float2 *mine = reinterpret_cast<const float2*>(lds) + ((pair >> 1) * TILES + (tile ^ (4 * (pair >> 1)))) * 2 + (pair & 1);
			float rows[2][6][4]; /* M A */
#pragma unroll
			for (int a = 0; a < 6; a++)
			{
				float m[2][6];
#pragma unroll
				for (int b = 0; b < 6; b++)
				{
					const float2 v = mine[(6 * a + b) * (8 * TILES * 2)];
					m[0][b] = v.x;
					m[1][b] = v.y;
				}
				output_line(m[0], rows[0][a]);
				output_line(m[1], rows[1][a]);
				__builtin_amdgcn_sched_barrier(0); /* not all 36 reads at once: the other half's products are still held */
			}
#pragma unroll
			for (int b = 0; b < 4; b++)
			{
				if (RESIDUAL && b + 1 < 4)
					load_residual(b + 1);
				float out[2][4];
#pragma unroll
				for (int e = 0; e < 2; e++)
				{
					const float m[6] = { rows[e][0][b], rows[e][1][b], rows[e][2][b], rows[e][3][b], rows[e][4][b], rows[e][5][b] };
					output_line(m, out[e]);
				}
#pragma unroll
				for (int a = 0; a < 4; a++)
				{
					const float v[2] = { out[0][a], out[1][a] };
					const float zv[2] = { RESIDUAL ? residual[b & 1][a].x : 0.0f, RESIDUAL ? residual[b & 1][a].y : 0.0f };
					float result[2];
					epi.template combine<RELU, RESIDUAL, 2>(result, v, columns, zv);
					const pair_t both = { result[0], result[1] };
					typedef unsigned int words_t __attribute__((ext_vector_type(2)));
					__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(words_t, both), ry, static_cast<int>(place(a, b)), 0, 0);
				}
			}
		}
	}

	/* U = G g G^T, G = [1 0 0; 2/3 2/3 2/3; 2/3 -2/3 2/3; 1/3 2/3 4/3; 1/3 -2/3 4/3; 0 0 2], in the order the kernel loads; filters and
	 * channels that fill its blocks are zeros */
	__device__ __forceinline__ void weight_line(float g0, float g1, float g2, float (&u)[6])
	{
		const float third = 1.0f / 3.0f, s = 2.0f * third * g0 + 2.0f * third * g2, q = third * g0 + 4.0f * third * g2, m = 2.0f * third * g1;
		u[0] = g0;
		u[1] = s + m;
		u[2] = s - m;
		u[3] = q + m;
		u[4] = q - m;
		u[5] = 2.0f * g2;
	}
	__global__ __launch_bounds__(256) void k_f4_weights(const float *__restrict__ w, float *__restrict__ U, int K, int C, int padded_c, int work, int invert)
	{
		const int id = blockIdx.x * 256 + threadIdx.x;
		if (id >= work)
			return;
		const int k = id / padded_c, c = id - k * padded_c;
		float taps[3][3];
#pragma unroll
		for (int i = 0; i < 3; i++)
#pragma unroll
			for (int j = 0; j < 3; j++)
			{
				const int tap = invert ? 8 - (3 * i + j) : 3 * i + j;
				taps[i][j] = k < K && c < C ? w[(static_cast<int64_t>(k) * 9 + tap) * C + c] : 0.0f;
			}
		float columns[3][6]; /* (G g)^T */
#pragma unroll
		for (int j = 0; j < 3; j++)
			weight_line(taps[0][j], taps[1][j], taps[2][j], columns[j]);
		const int slabs = padded_c / 8;
		float *to = U + (static_cast<int64_t>(k >> 5) * POINTS * slabs + (c >> 3)) * 256 + ((c & 7) >> 2) * 128 + (k & 31) * 4 + (c & 3);
#pragma unroll
		for (int i = 0; i < 6; i++)
		{
			float u[6];
			weight_line(columns[0][i], columns[1][i], columns[2][i], u);
#pragma unroll
			for (int j = 0; j < 6; j++)
				to[static_cast<int64_t>(6 * i + j) * slabs * 256] = u[j];
		}
	}

	int64_t padded_channels(int C)
	{
		return (static_cast<int64_t>(C) + CHANNELS - 1) / CHANNELS * CHANNELS;
	}
	int64_t padded_filters(int K)
	{
		return (static_cast<int64_t>(K) + FILTERS - 1) / FILTERS * FILTERS;
	}
	constexpr int64_t MOST_BYTES = 1ll << 29;
	int64_t pixels_of(const avhipConvShape &s)
	{
		return static_cast<int64_t>(s.N) * s.H * s.W;
	}
	int64_t tiles_of(const avhipConvShape &s)
	{
		return static_cast<int64_t>(s.N) * ((s.H + 3) / 4) * ((s.W + 3) / 4);
	}
}

namespace avhip
{
	bool winograd_f4_takes(const avhipConvShape &s, const void *x, const void *z, const void *y, double beta, int activation)
	{
		if (s.R != 3 || s.S != 3 || s.stride_h != 1 || s.stride_w != 1 || s.dil_h != 1 || s.dil_w != 1 || s.Ho != s.H || s.Wo != s.W
				|| !is_simple_activation(activation) || beta != 0.0 || s.K % 4 != 0 || !aligned_to(x, 4) || !aligned_to(y, 16)
				|| (z != nullptr && !aligned_to(z, 16)))
			return false;
		/* the output has the input's size, so every output pixel lies in a tile whatever the offset of the taps is */
		const int64_t blocks = (tiles_of(s) + TILES - 1) / TILES * (padded_filters(s.K) / FILTERS);
		return pixels_of(s) * s.C * 4 < MOST_BYTES && avhip_winograd_f4_weight_bytes(s.K, s.C) < MOST_BYTES && static_cast<int64_t>(s.C) * 4 * 8 < (1ll << 27)
				&& blocks * 512 < (1ll << 32) && pixels_of(s) * s.K * 4 < (1ll << 31) && s.pad_h >= -8 && s.pad_h <= 8 && s.pad_w >= -8 && s.pad_w <= 8;
	}
}

extern "C" int64_t avhip_winograd_f4_weight_bytes(int K, int C)
{
	return POINTS * padded_filters(K) * padded_channels(C) * 4;
}

extern "C" int avhip_winograd_f4_weight_transform(void *stream, int invert, const void *w, void *U, int K, int C)
{
	if (w == nullptr || U == nullptr || K <= 0 || C <= 0)
		return AVHIP_BAD_PARAM;
	if (avhip_winograd_f4_weight_bytes(K, C) >= MOST_BYTES)
		return AVHIP_NOT_SUPPORTED;
	const int padded_c = static_cast<int>(padded_channels(C)), work = static_cast<int>(padded_filters(K)) * padded_c;
	hipLaunchKernelGGL(k_f4_weights, dim3(ceil_div(work, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const float*>(w),
			static_cast<float*>(U), K, C, padded_c, work, invert != 0 ? 1 : 0);
	return 0;
}

extern "C" int avhip_conv2d_winograd_f4(void *stream, const avhipConvShape *shape, const void *x, const void *U, const void *bias, const void *z, void *y,
		double alpha1, double alpha2, double beta, int activation)
{
	if (shape == nullptr || x == nullptr || U == nullptr || y == nullptr)
		return AVHIP_BAD_PARAM;
	const avhipConvShape &s = *shape;
	if (s.N <= 0 || s.H <= 0 || s.W <= 0 || s.C <= 0 || s.K <= 0)
		return AVHIP_BAD_PARAM;
	if (!winograd_f4_takes(s, x, z, y, beta, activation) || !aligned_to(U, 16))
		return AVHIP_NOT_SUPPORTED;
	const int64_t tiles = tiles_of(s);
	const int64_t blocks = (tiles + TILES - 1) / TILES * (padded_filters(s.K) / FILTERS);
	F4Geom g;
	g.H = s.H;
	g.W = s.W;
	g.C = s.C;
	g.K = s.K;
	g.tiles = static_cast<int>(tiles);
	g.tiles_h = (s.H + 3) / 4;
	g.tiles_w = (s.W + 3) / 4;
	g.pad_h = s.pad_h;
	g.pad_w = s.pad_w;
	g.x_bytes = static_cast<unsigned int>(pixels_of(s) * s.C * 4);
	g.u_bytes = static_cast<unsigned int>(avhip_winograd_f4_weight_bytes(s.K, s.C));
	g.y_bytes = static_cast<unsigned int>(pixels_of(s) * s.K * 4);
	g.stages = static_cast<int>(padded_channels(s.C) / CHANNELS);
	g.filter_blocks = static_cast<int>(padded_filters(s.K) / FILTERS);
	const FloatEpilogue<float> epi { static_cast<const float*>(bias), static_cast<const float*>(z), static_cast<float*>(y), static_cast<float>(alpha1),
			static_cast<float>(alpha2), static_cast<float>(beta), activation, s.K, true };
	const bool relu = activation == ACT_RELU;
#define AVHIP_F4(RELU, RESIDUAL) hipLaunchKernelGGL((k_winograd_f4<RELU, RESIDUAL>), dim3(static_cast<unsigned int>(blocks)), dim3(512), 0, \
		static_cast<hipStream_t>(stream), static_cast<const float*>(x), static_cast<const float*>(U), g, epi)
	if (relu && z != nullptr)
		AVHIP_F4(true, true);
	else if (relu)
		AVHIP_F4(true, false);
	else if (z != nullptr)
		AVHIP_F4(false, true);
	else
		AVHIP_F4(false, false);
#undef AVHIP_F4
	return 0;
}

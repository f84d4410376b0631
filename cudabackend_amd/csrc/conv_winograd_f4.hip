/*
 * conv_winograd_f4.hip -- y = act(alpha1 * conv(x, w) + bias + alpha2 * z) + beta * y in fp32 by Winograd F(4x4, 3x3) in ONE kernel.
 *
 * The mathematics of the non-fused plan (src/winograd_nonfused.cu:257-519 of the reference, tables 534-575) without its matrices V and
 * M in memory: for 256 images of 15 x 15 with 128 channels these are 75 MB each, written and read once, and that traffic and not the
 * 4.8 GFLOP of the products was what bounded the plan (16 + 56 + 18 us).
 *
 * The products run on the bf16 matrix cores, which are sixteen times as fast as the fp32 ones: every value is cut into three bf16 pieces
 * (struct Pieces of mfma_core.hpp), and of the nine products of pieces the six that matter in 32 bits are taken.  A workgroup that finds sums which
 * are no numbers takes its tiles once more with fp32 products.
 *
 *   workgroup = 32 tiles (of 4 x 4 output pixels, in the order of the images) x 64 filters, eight wavefronts: four groups of nine
 *               transform points x two halves of the filters; a wavefront keeps its nine 32 x 32 products in 144 registers over the
 *               whole of k.  4096 tiles x 128 filters are 256 workgroups, one per compute unit;
 *   input     : per stage of 16 channels a work-item loads the 6 x 6 pixels of one tile and channel, transforms them in registers and
 *               writes them to LDS in pieces, two rows of points (a third) at a time into one of two buffers, in portions between the products of
 *               the third before;
 *   weights   : U in pieces and operand order (avhip_winograd_f4_weight_transform), one contiguous kilobyte per load, nine loads ahead;
 *   output    : M through LDS, 32 filters at a time, A^T M A in registers, the shared epilogue.
 *
 * What bounds it: a stage takes 4.1 us and its parts 1.6 (products, 3456 clocks), 1.4 (500 vector instructions of each of two wavefronts on a SIMD), 1.3
 * (LDS) and 2.2 (63 loads per wavefront) of them, one more in the way of the other than they should be with two wavefronts per SIMD;
 * around the stages 14 us of first loads, results and (one of them) the look at the sums.  All values of a stage must stay in registers: one in scratch makes every load in flight be
 * waited for (in-order counter), which cost a fifth.  The two passes of the output are a loop, for the same reason: written out they kept 24
 * registers in scratch and the kernel took 8 us longer.
 * Measured, fp32 products and now, one layer again and again: 256 x 15 x 15 x 128 -> 128 61 -> 47 us (three passes through memory 87), 64 channels 36 -> 25 us,
 * a tower of 20 of them in turn behind a first layer 1421 -> 1070 us (1050 with pieces cut off and not rounded, and sums not looked at: equal operands of 1 +
 * 2^-7 - 2^-23 then had an error of 4.7e-7, now below 2^-24, and those below 2^-110 lost their lower pieces).  Relative error against 64 bits 1.1e-6 to
 * 2.4e-6, with fp32 products 1.2e-6 to 2.9e-6.
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
	constexpr int PARTS = 3; /* of a stage: two rows of six points each, three of the twelve a wavefront's */
	constexpr int PART_POINTS = POINTS / PARTS, MY_PART = MY_POINTS / PARTS;
	/* V in LDS: [point of the part][piece][half of the channels][tile][channel of the half], bf16.  The halves lie 64 bytes more than their size apart,
	 * so that the sixteen channels of a tile go to different banks. */
	constexpr int V_HALF = TILES * 16 + 64, V_PIECE = 2 * V_HALF, V_POINT = 3 * V_PIECE, V_PART = PART_POINTS * V_POINT;

	struct F4Geom
	{
		int H, W, C, K, tiles, tiles_h, tiles_w, pad_h, pad_w;
		unsigned int x_bytes, u_bytes, y_bytes;
		int stages, filter_blocks;
	};

	/* A weight that has no pieces (an infinity, a NaN, or too large) is kept as this NaN and its own bits, the upper half first: its sums are NaN, and the
	 * workgroup that finds them takes the value from there. */
	constexpr unsigned int NO_PIECES = 0x7FC0u;
	constexpr float MOST_IN_PIECES = 0x1p127f;
	/* The highest piece of two values, as a pair; what is left of them in their place. */
	__device__ __forceinline__ unsigned int cut_pair(float (&value)[2])
	{
		typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
		const pair_t piece = { static_cast<__bf16>(value[0]), static_cast<__bf16>(value[1]) };
		unsigned int both = __builtin_bit_cast(unsigned int, piece);
		asm("" : "+v"(both)); /* or one of the two is converted a second time, alone */
		value[0] -= __builtin_bit_cast(float, both << 16);
		value[1] -= __builtin_bit_cast(float, both & 0xFFFF0000u);
		return both;
	}
	/* weight i of eight in pieces, as it was */
	__device__ __forceinline__ float joined(const Chunk (&u)[3], int i)
	{
		unsigned int bits[3];
#pragma unroll
		for (int n = 0; n < 3; n++)
		{
			const unsigned int pair = i < 2 ? u[n].u.x : i < 4 ? u[n].u.y : i < 6 ? u[n].u.z : u[n].u.w;
			bits[n] = i % 2 ? pair & 0xFFFF0000u : pair << 16;
		}
		const float sum = __builtin_bit_cast(float, bits[0]) + (__builtin_bit_cast(float, bits[1]) + __builtin_bit_cast(float, bits[2]));
		return bits[0] == NO_PIECES << 16 ? __builtin_bit_cast(float, bits[1] | bits[2] >> 16) : sum * (1.0f / PIECE_SCALE);
	}

	/* an offset beyond every tensor the launcher accepts (below 2^29 bytes), with the offset of a pixel added too */
	constexpr unsigned int NO_PIXEL = 0x80000000u;

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
	/* the same times PIECE_SCALE: a power of two, so that the results are those above in every bit, with three instructions more */
	__device__ __forceinline__ void scaled_input_line(float &d0, float &d1, float &d2, float &d3, float &d4, float &d5)
	{
		constexpr float S = PIECE_SCALE;
		const float a = d2 - 0.25f * d4, b = S * (d1 - 0.25f * d3), c = d4 - d2, e = S * (d3 - d1);
		const float o0 = S * ((d0 + 0.25f * c) - d2), o5 = (0.25f * S) * (d5 - d3) - e;
		d0 = o0;
		d1 = S * a + b;
		d2 = S * a - b;
		d3 = e + (0.5f * S) * c;
		d4 = (0.5f * S) * c - e;
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
		/* two parts of V; behind the loop M: [point][quad of filters][tile][filter of the quad], tiles in the order tile ^ 4 * quad: conflict-free
		 * for the work-items of neighbouring quads and for those of neighbouring tiles */
		constexpr int M_BYTES = POINTS * 32 * TILES * 4;
		static_assert(2 * V_PART <= M_BYTES, "the products of half of the filters take the place of the two parts");
		__shared__ __attribute__((aligned(16))) char lds[M_BYTES];
		__shared__ __attribute__((aligned(16))) int odd_waves[8];

		const int tid = threadIdx.x, lane = tid & 63;
		const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
		const int my_points = MY_PART * (wave & 3), my_half = wave >> 2; /* point q of part j is 12 j + my_points + q */
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
		/* which rows and columns of the tile exist: lane masks in scalar registers, of which there are enough */
		const unsigned int top = static_cast<unsigned int>(((image * g.H + 4 * th + g.pad_h) * g.W + 4 * tw + g.pad_w) * g.C + channel) * 4u;
		bool row[6], column[6];
#pragma unroll
		for (int a = 0; a < 6; a++)
		{
			const int ih = 4 * th + g.pad_h + a, iw = 4 * tw + g.pad_w + a;
			row[a] = t < g.tiles && ih >= 0 && ih < g.H;
			column[a] = iw >= 0 && iw < g.W;
		}
		const unsigned int pixel_bytes = static_cast<unsigned int>(g.C) * 4u, row_bytes = static_cast<unsigned int>(g.W) * pixel_bytes;
		const int last = g.stages - 1;
		const bool in_last = CHANNELS * last + channel < g.C;
		float d[36];
		auto load_row = [&](int stage, int a) __attribute__((always_inline))
		{
			const bool exists = row[a] && (stage < last || (stage == last && in_last)); /* (the stages behind the last: zeros) */
			unsigned int line = exists ? top + a * row_bytes + 64u * stage : NO_PIXEL;
			asm volatile("" : "+v"(line)); /* or 36 offsets are kept over the loop, more than there are registers */
#pragma unroll
			for (int b = 0; b < 6; b++)
				d[6 * a + b] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, static_cast<int>(column[b] ? line + b * pixel_bytes : NO_PIXEL), 0, 0));
		};
		/* (the sixteen channels of a tile are in the order 0, 8, 1, 9, .. in V and U) */
		const int put = ((channel & 7) >> 2) * V_HALF + tile * 16 + (channel & 3) * 4 + (channel >> 3) * V_POINT;
		auto transform_column = [&](int b) __attribute__((always_inline))
		{
			input_line(d[b], d[6 + b], d[12 + b], d[18 + b], d[24 + b], d[30 + b]);
		};
		auto transform_row = [&](int a) __attribute__((always_inline))
		{
			scaled_input_line(d[6 * a], d[6 * a + 1], d[6 * a + 2], d[6 * a + 3], d[6 * a + 4], d[6 * a + 5]);
		};
		/* Two values of V, in pieces.  Eight lanes beside the eight that have the first eight channels have the others of the
		 * same tile: they exchange values, so that each has both channels of a pair for one of the points, and write dwords: stores of single
		 * pieces took the LDS longer than the products take the matrix cores. */
		auto store_pieces = [&](int part, int buffer, int e) __attribute__((always_inline))
		{
			constexpr int ROW_ROTATE_8 = 0x128;
			const int e0 = __builtin_bit_cast(int, d[12 * part + e]), e1 = __builtin_bit_cast(int, d[12 * part + e + 1]);
			float value[2] = { __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(e0, e1, ROW_ROTATE_8, 15, 12, false)),
					__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(e1, e0, ROW_ROTATE_8, 15, 3, false)) };
			unsigned int *to = reinterpret_cast<unsigned int*>(lds + buffer * V_PART + put + e * V_POINT);
#pragma unroll
			for (int piece = 0; piece < 3; piece++)
				to[piece * V_PIECE / 4] = cut_pair(value);
		};
		/* A part is two rows of V: made in 18 pieces of work, one in front of each product of the part before; then their places in the
		 * registers are loaded with pixels of the next stage.  (Columns are transformed for the first part, as late as its work allows: its last
		 * pixels were requested a part ago.) */
		constexpr int SLOTS = 6 * MY_PART;
		static_assert(SLOTS == 18, "the work below");
		auto produce = [&](int slot, int part, int buffer, int next_stage) __attribute__((always_inline))
		{
			const int a = 2 * part;
			if (part == 0)
			{
				if (slot >= 4 && slot < 10)
					transform_column(slot - 4);
				if (slot == 10 || slot == 14)
					transform_row(a + (slot == 14 ? 1 : 0));
				if ((slot >= 11 && slot < 14) || slot >= 15)
				{
					const int e = slot < 14 ? 2 * (slot - 11) : 6 + 2 * (slot - 15);
					store_pieces(part, buffer, e);
				}
				if (slot == 14)
					load_row(next_stage, a);
				if (slot == 17)
					load_row(next_stage, a + 1);
			}
			else
			{
				if (slot == 0 || slot == 7)
					transform_row(a + (slot == 7 ? 1 : 0));
				if (slot < 7 && slot % 2 == 1)
					store_pieces(part, buffer, slot - 1);
				if (slot > 7 && slot < 14 && slot % 2 == 0)
					store_pieces(part, buffer, slot - 2);
				if (slot == 7)
					load_row(next_stage, a);
				if (slot == 14)
					load_row(next_stage, a + 1);
			}
		};

		/* U: [block of 32 filters][point][16 channels][piece][lane][8 channels] */
		const int u_first = ((2 * static_cast<int>(filter_block) + my_half) * POINTS + my_points) * g.stages;
		Chunk u[MY_PART][3];
		auto load_weights = [&](int stage, int part, int q) __attribute__((always_inline))
		{
			const int at = (u_first + (PART_POINTS * part + q) * g.stages + stage) * 3072;
#pragma unroll
			for (int piece = 0; piece < 3; piece++)
				u[q][piece].u = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ru, lane * 16, at + 1024 * piece, 0));
		};
		Mma<float>::acc_t acc[MY_POINTS]; /* [filters][tiles] */
		auto clear = [&]() __attribute__((always_inline))
		{
#pragma unroll
			for (int p = 0; p < MY_POINTS; p++)
#pragma unroll
				for (int v = 0; v < 16; v++)
					acc[p][v] = 0;
		};
		clear();
		const int r = lane & 31, half = lane >> 5;
		const int get = my_points * V_POINT + half * V_HALF + r * 16;
		/* One part: its products, v w of the pieces h + m + l with the smallest products first (what is left out, m l and below, is less than 2^-24 of
		 * the whole), and between them the work on the next part. */
		auto step = [&](int stage, int part, int buffer) __attribute__((always_inline))
		{
			constexpr int V_OF[6] = { 2, 1, 1, 0, 0, 0 }, U_OF[6] = { 0, 1, 0, 2, 1, 0 };
			const int next_part = (part + 1) % PARTS, next = part == PARTS - 1 ? stage + 1 : stage;
			const int weights_of = next < last ? next : last; /* (behind the last: its own once more) */
			__syncthreads(); /* this part of V is complete, the one before has been read */
			const char *from = lds + buffer * V_PART + get;
			Chunk cx[3];
			auto read = [&](int q, int piece) __attribute__((always_inline))
			{
				cx[piece].u = *reinterpret_cast<const uint4*>(from + q * V_POINT + piece * V_PIECE);
			};
			read(0, 2);
			read(0, 1);
			read(0, 0);
#pragma unroll
			for (int slot = 0; slot < SLOTS; slot++)
			{
				const int q = slot / 6, i = slot - 6 * q;
				produce(slot, next_part, buffer ^ 1, next + 1); /* (pixels behind the last channel: zeros) */
				__builtin_amdgcn_sched_barrier(0);
				Mma<bf16_t>::run(u[q][U_OF[i]], cx[V_OF[i]], acc[MY_PART * part + q]);
				__builtin_amdgcn_sched_barrier(0);
				if (q + 1 < MY_PART && (i == 0 || i == 2 || i == 5))
					read(q + 1, V_OF[i]);
				if (i == 5)
					load_weights(weights_of, next_part, q);
				__builtin_amdgcn_sched_barrier(0);
			}
		};

#pragma unroll
		for (int a = 0; a < 6; a++)
			load_row(0, a);
#pragma unroll
		for (int q = 0; q < MY_PART; q++)
			load_weights(0, 0, q);
#pragma unroll
		for (int slot = 0; slot < SLOTS; slot++)
			produce(slot, 0, 0, 1);
		for (int s = 0, odd = 0; s <= last; s++, odd ^= 1)
		{
			step(s, 0, odd);
			step(s, 1, odd ^ 1);
			step(s, 2, odd);
		}

		/* Sums that are no numbers, or so large that the output transform (which adds up to 361 of them) may leave the range of a float: an infinity, a NaN
		 * or a value that has no pieces is among the operands, or products reach 2^87.  The workgroup takes its tiles once more with fp32 products; so it
		 * does where alpha1 is so small that it cannot take the scale of the pieces back. */
		float size[4] = {}; /* finite if all sums are below 2^119 (comparisons hand their results to the scalar unit one by one, which took 0.6 us longer) */
#pragma unroll
		for (int p = 0; p < MY_POINTS; p++)
#pragma unroll
			for (int v = 0; v < 16; v++)
				size[v % 4] += 0x1p9f * __builtin_fabsf(acc[p][v]);
		const bool odd_wave = __builtin_amdgcn_ballot_w64(!((size[0] + size[1]) + (size[2] + size[3]) < __builtin_inff())) != 0
				|| (epi.alpha1 != 0.0f && __builtin_fabsf(epi.alpha1) < 0x1p-90f);
		if (lane == 0)
			odd_waves[wave] = odd_wave ? 1 : 0;
		__syncthreads();
		const int4 first_odd = *reinterpret_cast<const int4*>(odd_waves), last_odd = *reinterpret_cast<const int4*>(odd_waves + 4);
		const bool once_more = __builtin_amdgcn_readfirstlane(first_odd.x | first_odd.y | first_odd.z | first_odd.w | last_odd.x | last_odd.y | last_odd.z | last_odd.w) != 0;
		epi.alpha1 *= once_more ? 1.0f : 1.0f / (PIECE_SCALE * PIECE_SCALE);
		if (once_more)
		{
			clear();
			/* [point][channel, in the order of the weights][tile] */
			float *v_exact = reinterpret_cast<float*>(lds);
			const int place = 2 * (channel & 7) + (channel >> 3);
#pragma unroll 1
			for (int s = 0; s <= last; s++)
			{
#pragma unroll
				for (int a = 0; a < 6; a++)
					load_row(s, a);
#pragma unroll
				for (int b = 0; b < 6; b++)
					transform_column(b);
#pragma unroll
				for (int a = 0; a < 6; a++)
					input_line(d[6 * a], d[6 * a + 1], d[6 * a + 2], d[6 * a + 3], d[6 * a + 4], d[6 * a + 5]);
				__syncthreads();
#pragma unroll
				for (int p = 0; p < POINTS; p++)
					v_exact[(p * CHANNELS + place) * TILES + tile] = d[p];
				__syncthreads();
#pragma unroll
				for (int p = 0; p < MY_POINTS; p++)
				{
					const int point = PART_POINTS * (p / MY_PART) + my_points + p % MY_PART;
					load_weights(s, p / MY_PART, p % MY_PART);
#pragma unroll
					for (int i = 0; i < 8; i++)
						acc[p] = __builtin_amdgcn_mfma_f32_32x32x2f32(joined(u[p % MY_PART], i), v_exact[(point * CHANNELS + 8 * half + i) * TILES + r], acc[p], 0, 0, 0);
				}
			}
		}

		/* two filters of a tile per work-item: its place among 16 neighbours is the pair, so that runs of 128 bytes leave */
		const int pair = tid & 15;
		float4 *products = reinterpret_cast<float4*>(lds);
#pragma unroll 1
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
						products[((PART_POINTS * (p / MY_PART) + my_points + p % MY_PART) * 8 + quad) * TILES + (r ^ (4 * quad))] = make_float4(acc[p][4 * v], acc[p][4 * v + 1], acc[p][4 * v + 2], acc[p][4 * v + 3]);
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
	__global__ __launch_bounds__(256) void k_f4_weights(const float *__restrict__ w, unsigned short *__restrict__ U, int K, int C, int padded_c, int work, int invert)
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
		const int slabs = padded_c / CHANNELS, place = 2 * (c & 7) + ((c >> 3) & 1); /* in the order 0, 8, 1, 9, .. */
		unsigned short *to = U + (static_cast<int64_t>(k >> 5) * POINTS * slabs + c / CHANNELS) * 1536 + ((place >> 3) * 256) + (k & 31) * 8 + (place & 7);
#pragma unroll
		for (int i = 0; i < 6; i++)
		{
			float u[6];
			weight_line(columns[0][i], columns[1][i], columns[2][i], u);
#pragma unroll
			for (int j = 0; j < 6; j++)
			{
				unsigned short *piece = to + static_cast<int64_t>(6 * i + j) * slabs * 1536;
				float rest[2] = { u[j] * PIECE_SCALE, 0.0f };
				const unsigned int bits = __builtin_bit_cast(unsigned int, u[j]);
				const bool whole = fabsf(rest[0]) >= MOST_IN_PIECES || !(fabsf(u[j]) < INFINITY);
#pragma unroll
				for (int n = 0; n < 3; n++)
				{
					const unsigned int cut = cut_pair(rest);
					piece[512 * n] = static_cast<unsigned short>(!whole ? cut : n == 0 ? NO_PIECES : n == 1 ? bits >> 16 : bits);
				}
			}
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
	constexpr int64_t MOST_BYTES = 1ll << 29, MOST_WEIGHT_BYTES = 3ll << 28;
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
		return pixels_of(s) * s.C * 4 < MOST_BYTES && avhip_winograd_f4_weight_bytes(s.K, s.C) < MOST_WEIGHT_BYTES && static_cast<int64_t>(s.C) * 4 * 8 < (1ll << 27)
				&& blocks * 512 < (1ll << 32) && pixels_of(s) * s.K * 4 < (1ll << 31) && s.pad_h >= -8 && s.pad_h <= 8 && s.pad_w >= -8 && s.pad_w <= 8;
	}
}

extern "C" int64_t avhip_winograd_f4_weight_bytes(int K, int C)
{
	return POINTS * padded_filters(K) * padded_channels(C) * 6;
}

extern "C" int avhip_winograd_f4_weight_transform(void *stream, int invert, const void *w, void *U, int K, int C)
{
	if (w == nullptr || U == nullptr || K <= 0 || C <= 0)
		return AVHIP_BAD_PARAM;
	if (avhip_winograd_f4_weight_bytes(K, C) >= MOST_WEIGHT_BYTES)
		return AVHIP_NOT_SUPPORTED;
	const int padded_c = static_cast<int>(padded_channels(C)), work = static_cast<int>(padded_filters(K)) * padded_c;
	hipLaunchKernelGGL(k_f4_weights, dim3(ceil_div(work, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const float*>(w),
			static_cast<unsigned short*>(U), K, C, padded_c, work, invert != 0 ? 1 : 0);
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

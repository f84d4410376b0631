/*
 * gemm_tn.hip -- C[b] = alpha * A[b]^T B[b] + beta * C[b] on the matrix cores: the product of the Winograd weight gradient,
 * where k runs over the tiles of the batch (hundreds to tens of thousands), C is one K x C matrix per transform point
 * (16 or 36 of them) and both operands are contiguous along m and n, not along k.
 *
 * No transpose is made.  For fp32 the operand layout of v_mfma_f32_32x32x2_f32 (lane l: row l % 32, k l / 32) is exactly a
 * coalesced load of two rows of A, and the eight k that a lane has of a stage are an operand of a bf16 product too: with tiles of 64 x 64 the
 * values are cut into three bf16 pieces in registers (struct Pieces of mfma_core.hpp), and six of the nine products of pieces are taken.  (The cutting costs
 * as much as the products save with 32 x 32: 12.6 against 11.4 us below.)  For 16-bit types a lane loads one dword (two neighbouring m) of four or eight
 * k rows and separates them with v_perm_b32 into the operand chunks of two MFMA tiles, one of the even and one of the odd m, or exchanges one
 * of the two with the sixteen lanes beside it; what cannot be read in pairs (odd sizes) is loaded element by element.  k rows and m, n
 * outside the matrices come back as zeros from the buffer loads, so the loop has no branch.
 *
 * Workgroup = 8 wavefronts on ONE tile of C (64 x 64 or 32 x 32): each takes every eighth stage of 16 k rows, two to four
 * stages in flight in registers, nothing shared in the loop and no barrier; the eight partial tiles are added through LDS at
 * the end, in a fixed order.  The split along k inside the workgroup is what fills the chip: a gradient of 128 x 128
 * channels has 144 tiles of 64 x 64 (F(4x4, 3x3)), 1152 wavefronts for 1024 SIMDs.  Sixteen wavefronts on a tile of 32 x 32 were slower at every size.
 *
 * Measured (36 products 128 x 128 over k = 512, fp32, operands from L2 / the last-level cache): 9.8 us, of which the
 * 18.9 MB of operands need 3.4 and the matrix cores 1.5; 11.4 with fp32 products, 74 in the generic kernel.  16-bit, tiles of 32 x 32, pairs against single
 * elements: 16 products 72 x 96 over 15561 43.1 -> 38.7 us, 32 x 32 over 4608 12.2 -> 8.4, 64 x 80 over 750 5.9 -> 4.6.  What bounds it at small
 * sizes is the chain of one launch: first loads, one or two waves of MFMAs, the sum through LDS.  With a last round that requested as many stages again and multiplied zeros to its end,
 * 120 drawn gradients took 4.5 % longer, all launches.  fp32 values loaded in pairs (half as many loads, sixteen lanes exchanged for 32 x 32) took 7 to 12 % longer.
 */
#include <cmath>
#include <type_traits>

#include "gemm_tn.hpp"
#include "mfma_core.hpp"

namespace
{
	using namespace avhip;

	constexpr int WAVES = 8;
	constexpr int STAGE = 16; /* k rows of one stage */

	struct TnGeom
	{
		int M, N, K, row_tiles, col_tiles;
		unsigned int a_pitch, b_pitch; /* bytes between k rows */
		unsigned int a_extent, b_extent; /* bytes of one batch entry */
		int ldc;
		int64_t a_batch, b_batch, c_batch; /* elements */
		float alpha, beta;
	};

	/* The 16 k rows of one operand that a wavefront holds for one stage: T MFMA tiles of 32 rows.  PAIRS (16-bit types): a lane loads two neighbouring
	 * elements at once; tile t of two holds the elements 2 * (lane % 32) + t of the 64, one tile alone the even ones in lanes 0 to 15 and the odd ones
	 * in 16 to 31.  Otherwise tile t holds 32 t + lane % 32. */
	template<typename TE, int T, bool PAIRS>
	struct Operand
	{
		static constexpr bool WIDE = sizeof(TE) == 4, ONE_OF_PAIRS = PAIRS && T == 1;
		static constexpr int ROWS = ONE_OF_PAIRS ? 4 : 8; /* loads of a lane for one tile or pair of tiles, of one k row each */
		static constexpr int WORDS = PAIRS ? ROWS : 8 * T;
		unsigned int v[WORDS];
		__device__ static __forceinline__ int element(int tile, int r)
		{
			return ONE_OF_PAIRS ? 2 * (r & 15) + (r >> 4) : PAIRS ? 2 * r + tile : 32 * tile + r;
		}
		/* byte offset of this lane's element in its load j of a stage */
		__device__ static __forceinline__ unsigned int origin(int first, unsigned int pitch, int lane, int j)
		{
			const unsigned int half = lane >> 5;
			if (ONE_OF_PAIRS) /* four k rows a load */
				return (4 * j + (lane >> 4)) * pitch + (first + 2 * (lane & 15)) * sizeof(TE);
			return (WIDE ? 2 * j + half : j + 8 * half) * pitch + (first + element(0, lane & 31)) * sizeof(TE);
		}
		__device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t rsrc, const unsigned int (&rows)[ROWS])
		{
#pragma unroll
			for (int j = 0; j < ROWS; j++)
			{
				if constexpr (WIDE)
				{
#pragma unroll
					for (int t = 0; t < T; t++)
						v[j * T + t] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, static_cast<int>(rows[j] + t * 128), 0, 0);
				}
				else if constexpr (PAIRS)
					v[j] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, static_cast<int>(rows[j]), 0, 0);
				else
				{
#pragma unroll
					for (int t = 0; t < T; t++)
						v[j * T + t] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, static_cast<int>(rows[j] + t * 64), 0, 0);
				}
			}
		}
		/* 16-bit types: the operand chunk (8 consecutive k) of tile t */
		__device__ __forceinline__ Chunk chunk(int t) const
		{
			unsigned int w[4];
			if constexpr (ONE_OF_PAIRS)
			{
				/* sixteen lanes keep the even elements and take those of their neighbours' k rows, which keep the odd ones */
#pragma unroll
				for (int q = 0; q < 2; q++)
				{
					const auto s = __builtin_amdgcn_permlane16_swap(__builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], 0x05040100u),
							__builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], 0x07060302u), false, false);
					w[2 * q] = s[0];
					w[2 * q + 1] = s[1];
				}
			}
			else
			{
#pragma unroll
				for (int q = 0; q < 4; q++)
				{
					if constexpr (PAIRS)
						w[q] = __builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], t ? 0x07060302u : 0x05040100u);
					else
						w[q] = (v[(2 * q) * T + t] & 0xFFFFu) | (v[(2 * q + 1) * T + t] << 16);
				}
			}
			Chunk c;
			c.u = make_uint4(w[0], w[1], w[2], w[3]);
			return c;
		}
		/* fp32: the eight values of tile t */
		__device__ __forceinline__ void cut(int t, Pieces &pieces) const
		{
#pragma unroll
			for (int q = 0; q < 4; q++)
				pieces.cut(q, PIECE_SCALE * __builtin_bit_cast(float, v[(2 * q) * T + t]), PIECE_SCALE * __builtin_bit_cast(float, v[(2 * q + 1) * T + t]));
		}
	};

	template<typename TE, typename TC, int T, bool PAIRS>
	__global__ __launch_bounds__(64 * WAVES, 2) void k_gemm_tn(const TE *__restrict__ A, const TE *__restrict__ B, TC *C, TnGeom g)
	{
		typedef Operand<TE, T, PAIRS> Op;
		constexpr int SIDE = 32 * T;
		constexpr int QUADS = T * T * 4; /* 16-byte runs a lane holds of the tile */
		constexpr int DEPTH = T == 1 ? 4 : Op::WIDE ? 2 : 3; /* stages in flight */
		typedef float quad_t __attribute__((ext_vector_type(4)));
		__shared__ quad_t sums[4][QUADS][64];

		const int lane = threadIdx.x & 63;
		const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
		/* the tiles of a batch entry share its rows: a contiguous run of them goes to one XCD and its L2 */
		const int tile = static_cast<int>(xcd_block(blockIdx.x, gridDim.x));
		const int per_entry = g.row_tiles * g.col_tiles;
		const int batch = tile / per_entry, in_entry = tile - batch * per_entry;
		const int m0 = (in_entry / g.col_tiles) * SIDE, n0 = (in_entry % g.col_tiles) * SIDE;
		const char *a = reinterpret_cast<const char*>(A + batch * g.a_batch);
		const char *b = reinterpret_cast<const char*>(B + batch * g.b_batch);

		unsigned int rows_a[Op::ROWS], rows_b[Op::ROWS];
#pragma unroll
		for (int j = 0; j < Op::ROWS; j++)
		{
			rows_a[j] = Op::origin(m0, g.a_pitch, lane, j);
			rows_b[j] = Op::origin(n0, g.b_pitch, lane, j);
		}
		/* the descriptor moves with the stage and shrinks to what is left of the matrix: nothing, behind the last stage */
		auto remaining = [](const char *base, unsigned int extent, int64_t skip)
		{
			return make_buffer(base + skip, skip < extent ? extent - static_cast<unsigned int>(skip) : 0u);
		};
		Op oa[DEPTH], ob[DEPTH];
		auto fetch = [&](int d, int stage) __attribute__((always_inline))
		{
			oa[d].fetch(remaining(a, g.a_extent, static_cast<int64_t>(stage) * STAGE * g.a_pitch), rows_a);
			ob[d].fetch(remaining(b, g.b_extent, static_cast<int64_t>(stage) * STAGE * g.b_pitch), rows_b);
		};
		f32x16_t acc[T][T];
		auto multiply = [&](const Op &x, const Op &y, auto exact) __attribute__((always_inline))
		{
			if constexpr (Op::WIDE && (T == 1 || exact.value))
			{
#pragma unroll
				for (int p = 0; p < 8; p++)
#pragma unroll
					for (int i = 0; i < T; i++)
#pragma unroll
						for (int j = 0; j < T; j++)
							acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, x.v[p * T + i]), __builtin_bit_cast(float, y.v[p * T + j]),
									acc[i][j], 0, 0, 0);
			}
			else if constexpr (Op::WIDE)
			{
				Pieces ca[T];
#pragma unroll
				for (int i = 0; i < T; i++)
					x.cut(i, ca[i]);
#pragma unroll
				for (int j = 0; j < T; j++)
				{
					Pieces cb;
					y.cut(j, cb);
#pragma unroll
					for (int p = 0; p < PIECE_PRODUCTS; p++)
#pragma unroll
						for (int i = 0; i < T; i++)
							Mma<bf16_t>::run(ca[i].p[PIECE_OF_A[p]], cb.p[PIECE_OF_B[p]], acc[i][j]);
				}
			}
			else
			{
				Chunk ca[T], cb[T];
#pragma unroll
				for (int i = 0; i < T; i++)
				{
					ca[i] = x.chunk(i);
					cb[i] = y.chunk(i);
				}
#pragma unroll
				for (int i = 0; i < T; i++)
#pragma unroll
					for (int j = 0; j < T; j++)
						Mma<TE>::run(ca[i], cb[j], acc[i][j]);
			}
		};

		const int stages = (g.K + STAGE - 1) / STAGE;
		const int mine = (stages - wave + WAVES - 1) / WAVES; /* stages wave, wave + 8, ... */
		auto walk = [&](auto exact) __attribute__((always_inline))
		{
#pragma unroll
			for (int i = 0; i < T; i++)
#pragma unroll
				for (int j = 0; j < T; j++)
#pragma unroll
					for (int v = 0; v < 16; v++)
						acc[i][j][v] = 0.0f;
#pragma unroll
			for (int d = 0; d < DEPTH; d++)
				fetch(d, wave + d * WAVES);
			int left = mine; /* may be none */
			for (int next = wave + DEPTH * WAVES; left > DEPTH; left -= DEPTH, next += DEPTH * WAVES)
			{
#pragma unroll
				for (int d = 0; d < DEPTH; d++)
				{
					multiply(oa[d], ob[d], exact);
					fetch(d, next + d * WAVES); /* zeros behind the last stage */
				}
			}
			/* the last round requests nothing, and multiplies what there is */
#pragma unroll
			for (int d = 0; d < DEPTH; d++)
				if (d < left)
					multiply(oa[d], ob[d], exact);
		};
		walk(std::false_type());
		if constexpr (Op::WIDE && T == 2)
		{
			/* sums that are no numbers: this wavefront's share of k once more with fp32 products, whatever these give (struct Pieces) */
			if (__builtin_amdgcn_ballot_w64(!finish_pieces(acc)) != 0)
				walk(std::true_type());
		}

		/* eight partial tiles: 4..7 onto 0..3 in registers, then every wavefront adds its share of the four copies */
		auto write = [&](int copy) __attribute__((always_inline))
		{
#pragma unroll
			for (int t = 0; t < T * T; t++)
#pragma unroll
				for (int i = 0; i < 4; i++)
				{
					const f32x16_t &v = acc[t / T][t % T];
					sums[copy][t * 4 + i][lane] = quad_t { v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3] };
				}
		};
		if (wave >= 4)
			write(wave - 4);
		__syncthreads();
		if (wave < 4)
		{
#pragma unroll
			for (int t = 0; t < T * T; t++)
#pragma unroll
				for (int i = 0; i < 4; i++)
				{
					const quad_t o = sums[wave][t * 4 + i][lane];
#pragma unroll
					for (int e = 0; e < 4; e++)
						acc[t / T][t % T][4 * i + e] += o[e];
				}
			write(wave); /* each wavefront its own copy, just read by itself */
		}
		__syncthreads();
		TC *c = C + batch * g.c_batch;
		constexpr int SHARE = QUADS >= WAVES ? QUADS / WAVES : 1;
#pragma unroll
		for (int h = 0; h < SHARE; h++)
		{
			/* T == 2: the two column tiles of one row group, so that both halves of a pair of columns leave from one lane */
			const int q = T == 2 ? ((wave >> 2) * 2 + h) * 4 + (wave & 3) : wave;
			if (q < QUADS)
			{
				quad_t total = sums[0][q][lane];
#pragma unroll
				for (int copy = 1; copy < 4; copy++)
					total += sums[copy][q][lane];
				const int n = n0 + Op::element((q / 4) % T, lane & 31);
#pragma unroll
				for (int e = 0; e < 4; e++)
				{
					const int m = m0 + Op::element((q / 4) / T, 8 * (q & 3) + 4 * (lane >> 5) + e);
					if (m < g.M && n < g.N)
					{
						TC *p = c + static_cast<size_t>(m) * g.ldc + n;
						float v = g.alpha * total[e];
						if (g.beta != 0.0f)
							v += g.beta * static_cast<float>(Traits<TC>::load(*p));
						*p = Traits<TC>::store(v);
					}
				}
			}
		}
	}
}

namespace
{
	/* The side of a tile of C: 32 while tiles of 64 leave the chip short of work.  16-bit types are bound by their operand loads, which large tiles halve
	 * (at 64 large tiles 18 to 54 % slower than small ones, at 160 to 256 equal, above faster).  fp32: small tiles have fp32 products and four of
	 * them share a compute unit, large ones have bf16 pieces and a compute unit each, so that 288 of them are two rounds and cost what 512 do.
	 * Microseconds of the two, fitted to 115 products with both (16 or 36 of 32 to 256 a side over 60 to 7128; root mean square error 10 and 7 %);
	 * with the large ones 5 % below, the one taken is 0.2 % slower than the faster one on average and 7 % at most (80 x 224 over 2150, 36 of them, 288 large tiles:
	 * 54.7 : 36.6 us, 216 x 32 over 1716 22.7 : 15.5; 128 x 128 over 512, 144 large tiles 9.8 : 11.4, 168 x 128 over 273, 216 8.5 : 14.1). */
	int tn_side(int element_bytes, int batch, int M, int N, int K)
	{
		auto tiles = [&](int side) { return static_cast<int64_t>(ceil_div(M, side)) * ceil_div(N, side) * batch; };
		if (element_bytes != 4)
			return tiles(64) < 128 ? 32 : 64;
		if (tiles(32) * 64 * WAVES >= (1ll << 32)) /* more work-items than a launch takes along one direction */
			return 64;
		const int stages = static_cast<int>(ceil_div(ceil_div(K, STAGE), WAVES)); /* of a wavefront; large tiles have them in flight in pairs */
		auto on_a_unit = [&](int side) { return std::ceil(static_cast<double>(tiles(side)) / 256.0); };
		const double small = 2.4 + on_a_unit(32) * (1.8 + 0.51 * stages), large = 0.7 + on_a_unit(64) * (4.1 + 0.86 * stages + 0.80 * ((stages + 1) / 2));
		return large < 0.95 * small ? 64 : 32;
	}
}

extern "C" int avhip_gemm_tn_side(int element_bytes, int batch, int M, int N, int K)
{
	return tn_side(element_bytes, batch, M, N, K);
}

namespace avhip
{
	template<typename TE, typename TC>
	bool gemm_tn_launch(hipStream_t stream, const void *A, const void *B, void *C, int batch, int M, int N, int K, int lda, int ldb, int ldc, int64_t strideA,
			int64_t strideB, int64_t strideC, float alpha, float beta)
	{
		constexpr int64_t SZ = sizeof(TE);
		const int64_t a_extent = (static_cast<int64_t>(K - 1) * lda + M) * SZ, b_extent = (static_cast<int64_t>(K - 1) * ldb + N) * SZ;
		/* offsets within a stage are 32-bit and the loop may point a few stages behind the end */
		if (a_extent >= (1ll << 31) || b_extent >= (1ll << 31) || lda >= (1 << 22) || ldb >= (1 << 22) || lda < M || ldb < N)
			return false;
		TnGeom g;
		g.M = M;
		g.N = N;
		g.K = K;
		g.a_pitch = static_cast<unsigned int>(lda * SZ);
		g.b_pitch = static_cast<unsigned int>(ldb * SZ);
		g.a_extent = static_cast<unsigned int>(a_extent);
		g.b_extent = static_cast<unsigned int>(b_extent);
		g.ldc = ldc;
		g.a_batch = strideA;
		g.b_batch = strideB;
		g.c_batch = strideC;
		g.alpha = alpha;
		g.beta = beta;
		const int side = tn_side(SZ, batch, M, N, K);
		const bool small = side == 32;
		g.row_tiles = static_cast<int>(ceil_div(M, side));
		g.col_tiles = static_cast<int>(ceil_div(N, side));
		const int64_t tiles = static_cast<int64_t>(g.row_tiles) * g.col_tiles * batch;
		if (tiles * 64 * WAVES >= (1ll << 32)) /* more work-items than a launch takes along one direction */
			return false;
		const dim3 grid(static_cast<unsigned int>(tiles)), block(64 * WAVES);
		const TE *a = static_cast<const TE*>(A), *b = static_cast<const TE*>(B);
		TC *c = static_cast<TC*>(C);
		if constexpr (sizeof(TE) == 2)
		{
			/* pairs: every dword of a row aligned and inside it */
			const bool pairs = M % 2 == 0 && N % 2 == 0 && lda % 2 == 0 && ldb % 2 == 0 && strideA % 2 == 0 && strideB % 2 == 0 && aligned_to(A, 4) && aligned_to(B, 4);
			if (pairs)
			{
				if (small)
					hipLaunchKernelGGL((k_gemm_tn<TE, TC, 1, true>), grid, block, 0, stream, a, b, c, g);
				else
					hipLaunchKernelGGL((k_gemm_tn<TE, TC, 2, true>), grid, block, 0, stream, a, b, c, g);
				return true;
			}
		}
		if (small)
			hipLaunchKernelGGL((k_gemm_tn<TE, TC, 1, false>), grid, block, 0, stream, a, b, c, g);
		else
			hipLaunchKernelGGL((k_gemm_tn<TE, TC, 2, false>), grid, block, 0, stream, a, b, c, g);
		return true;
	}

#define AVHIP_INSTANTIATE(TE, TC) template bool gemm_tn_launch<TE, TC>(hipStream_t, const void*, const void*, void*, int, int, int, int, int, int, int, int64_t, int64_t, int64_t, float, float);
	AVHIP_INSTANTIATE(float, float)
	AVHIP_INSTANTIATE(f16_t, f16_t)
	AVHIP_INSTANTIATE(f16_t, float)
	AVHIP_INSTANTIATE(bf16_t, bf16_t)
	AVHIP_INSTANTIATE(bf16_t, float)
#undef AVHIP_INSTANTIATE
}

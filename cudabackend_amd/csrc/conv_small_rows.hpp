/*
 * conv_small_rows.hpp -- how the kernels of small tiles (conv_small.hip, conv_small16.hip) load rows of channels that are no whole number of 16-byte chunks.
 */
#ifndef AVHIP_CONV_SMALL_ROWS_HPP_
#define AVHIP_CONV_SMALL_ROWS_HPP_

#include "mfma_core.hpp"

namespace avhip
{
	/* What the rows of channels (one pixel, one tap of a filter) are known to be: whole 16-byte chunks; dwords; elements. */
	constexpr int ROWS_OF_CHUNKS = 0, ROWS_OF_DWORDS = 1, ROWS_OF_ELEMENTS = 2;

	/* 16 bytes on their way from memory, from any byte on if ROW is ROWS_OF_ELEMENTS: then they are the aligned dwords around them */
	template<int ROW>
	struct Piece
	{
		uint4 u;
		__device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t rsrc, unsigned int offset)
		{
			u = buffer_fetch(rsrc, offset);
		}
		/* what belongs to the row: `left` bytes of it from the first one on */
		__device__ __forceinline__ uint4 get(unsigned int, const uint4 &keep) const
		{
			if (ROW == ROWS_OF_CHUNKS)
				return u;
			return make_uint4(u.x & keep.x, u.y & keep.y, u.z & keep.z, u.w & keep.w);
		}
	};
	template<>
	struct Piece<ROWS_OF_ELEMENTS>
	{
		uint4 u;
		unsigned int next;
		__device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t rsrc, unsigned int offset)
		{
			u = buffer_fetch(rsrc, offset & ~3u);
			next = __builtin_amdgcn_raw_buffer_load_b32(rsrc, static_cast<int>((offset & ~3u) + 16), 0, 0);
		}
		__device__ __forceinline__ uint4 get(unsigned int offset, const uint4 &keep) const
		{
			return make_uint4(__builtin_amdgcn_alignbyte(u.y, u.x, offset & 3) & keep.x, __builtin_amdgcn_alignbyte(u.z, u.y, offset & 3) & keep.y,
					__builtin_amdgcn_alignbyte(u.w, u.z, offset & 3) & keep.z, __builtin_amdgcn_alignbyte(next, u.w, offset & 3) & keep.w);
		}
	};
	/* which bits of a dword belong to a row that has `left` more bytes */
	__device__ __forceinline__ unsigned int keep_bits(int left)
	{
		return left >= 4 ? ~0u : left <= 0 ? 0u : (1u << (8 * left)) - 1;
	}
}

#endif /* AVHIP_CONV_SMALL_ROWS_HPP_ */

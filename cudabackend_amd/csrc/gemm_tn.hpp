/*
 * gemm_tn.hpp -- internal interface of the matrix-core kernel for C = alpha * A^T B + beta * C (gemm_tn.hip).
 */
#ifndef AVHIP_GEMM_TN_HPP_
#define AVHIP_GEMM_TN_HPP_

#include "common.hpp"

extern "C"
{
	/* The side of the tiles of C that a product is taken in, 32 or 64 (fp32: the latter in bf16 pieces).  Exported for tests. */
	AVHIP_API int avhip_gemm_tn_side(int element_bytes, int batch, int M, int N, int K);
}

namespace avhip
{
	/* Launches the (T, N) product C[b][m][n] = alpha * sum_k A[b][k][m] * B[b][k][n] + beta * C[b][m][n] (row-major, fp32
	 * accumulation) and returns true; returns false without side effects when a batch entry of A or B is 2 GiB or larger. */
	template<typename TE, typename TC>
	bool gemm_tn_launch(hipStream_t stream, const void *A, const void *B, void *C, int batch, int M, int N, int K, int lda, int ldb, int ldc, int64_t strideA,
			int64_t strideB, int64_t strideC, float alpha, float beta);
}

#endif /* AVHIP_GEMM_TN_HPP_ */

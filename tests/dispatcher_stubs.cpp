/*
 * dispatcher_stubs.cpp -- stands in for the HIP runtime and the kernel layer, so that the dispatcher of backend.cpp runs on a machine
 * without a GPU: "device" memory is host memory, launchers count their calls and compute nothing.  Linked with backend.cpp by
 * test_dispatcher_host.py.
 */
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "../cudabackend_amd/csrc/conv_estimates.hpp"
#include "../cudabackend_amd/csrc/conv_winograd_f4.hpp"

namespace
{
	std::map<std::string, int> calls;
	bool malloc_fails = false, capturing = false;
	int strided_workgroups = 0;
	double ring_us = 0.0, direct_us = 0.0;
	int called(const char *name, int result = 0)
	{
		calls[name]++;
		return result;
	}
}

extern "C"
{
	AVHIP_API void stub_set(int malloc_fails_now, int capturing_now)
	{
		malloc_fails = malloc_fails_now != 0;
		capturing = capturing_now != 0;
		calls.clear();
	}
	/* the parity-plane kernel's workgroups (0: it takes nothing) and what the ring kernel answers for every layer (0: it takes nothing) */
	AVHIP_API void stub_set_strided(int workgroups, double ring_us_now)
	{
		strided_workgroups = workgroups;
		ring_us = ring_us_now;
	}
	/* what direct sums are estimated to take, for every layer (0: not weighed) */
	AVHIP_API void stub_set_direct(double direct_us_now)
	{
		direct_us = direct_us_now;
	}
	AVHIP_API int stub_calls(const char *name)
	{
		return calls[name];
	}

	hipError_t hipMalloc(void **p, size_t bytes)
	{
		if (malloc_fails)
			return hipErrorOutOfMemory;
		*p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096); /* never touched by the launchers below */
		return hipSuccess;
	}
	hipError_t hipFree(void *p)
	{
		std::free(p);
		return hipSuccess;
	}
	hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
	hipError_t hipGetDevice(int *n) { *n = 0; return hipSuccess; }
	hipError_t hipSetDevice(int) { return hipSuccess; }
	hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) { std::memset(p, 0, sizeof(*p)); return hipSuccess; }
	hipError_t hipGetLastError() { return hipSuccess; }
	hipError_t hipGetSymbolAddress(void **p, const void*) { static double scratch[64]; *p = scratch; return hipSuccess; }
	hipError_t hipDeviceSynchronize() { return hipSuccess; }
	hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
	hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
	hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
	hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
	hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
	hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
	hipError_t hipStreamCreate(hipStream_t *s) { *s = reinterpret_cast<hipStream_t>(8); return hipSuccess; }
	hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
	hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
	{
		*s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
		return hipSuccess;
	}
	hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
	hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
	hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
	hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }

	int avhip_conv2d_split_k_workspace(int, const avhipConvShape*, int64_t *bytes) { *bytes = 0; return 0; }
	int64_t avhip_winograd_f4_weight_bytes(int K, int C) { return 144ll * K * C; }
	int avhip_winograd_f4_weight_transform(void*, int, const void*, void*, int, int) { return called("f4_weights"); }
	int avhip_conv2d_winograd_f4(void*, const avhipConvShape*, const void*, const void*, const void*, const void*, void*, double, double, double, int)
	{
		return called("f4");
	}
	int avhip_winograd_weight_transform(void*, int, int, int, int, int, const void*, void*, int, int) { return called("weights"); }
	int avhip_winograd_input_transform(void*, int, int, int, int, const void*, void*, int, int, int, int, int, int, const void*) { return called("input_transform"); }
	int avhip_gemm_batched(void*, int, int, int, int, const void*, const void*, void*, int, int, int, int, int, int, int, int64_t, int64_t, int64_t, double, double)
	{
		return called("gemm");
	}
	int avhip_winograd_output_transform(void*, int, int, int, int, const void*, void*, const void*, const void*, int, int, int, int, double, double, double, int)
	{
		return called("output_transform");
	}
	int avhip_conv2d_implicit_gemm(void*, int, int, int, const avhipConvShape*, const void*, const void*, const void*, const void*, void*, const void*, double,
			double, double, int, const float*)
	{
		return called("implicit_gemm");
	}
	int avhip_conv2d_winograd_rows_plan(int, const avhipConvShape*, int*, int*) { return AVHIP_NOT_SUPPORTED; }
	int avhip_conv2d_strided_plan(int, const avhipConvShape*, int *workgroups, int *rows_used)
	{
		*workgroups = strided_workgroups;
		*rows_used = 224;
		return strided_workgroups > 0 ? 0 : AVHIP_NOT_SUPPORTED;
	}
	int64_t avhip_conv2d_strided_weight_bytes(int K, int C) { return 18ll * K * C; }
	int avhip_conv2d_strided_weight_layout(void*, int, int, const void*, void*, int, int) { return called("strided_weights"); }
	int avhip_conv2d_strided(void*, int, const avhipConvShape*, const void*, const void*, const void*, const void*, void*, double, double, double, int)
	{
		return called("strided");
	}
	double avhip_conv2d_ring_us(int, int, const avhipConvShape*, int, int) { return ring_us; }
	double avhip_conv2d_small_us(int, const avhipConvShape*, int) { return direct_us; }
	int avhip_conv2d_winograd_fused(void*, int, const avhipConvShape*, const void*, const void*, const void*, const void*, void*, double, double, double, int)
	{
		return called("fused");
	}
	int avhip_conv2d_pointwise_block_plan(int, const avhipConvShape*, int*, int*) { return AVHIP_NOT_SUPPORTED; }
}

/* never reached by the calls of the test: AVHIP_NOT_SUPPORTED */
#define STUB_UNUSED(name) asm(".text\n.globl " #name "\n.type " #name ",@function\n" #name ":\n\tmovl $-1, %eax\n\tret\n");
STUB_UNUSED(avhip_add_bias)
STUB_UNUSED(avhip_affine_forward)
STUB_UNUSED(avhip_batchnorm_inference)
STUB_UNUSED(avhip_change_type)
STUB_UNUSED(avhip_conv2d_implicit_gemm_split_k)
STUB_UNUSED(avhip_conv2d_pointwise_block)
STUB_UNUSED(avhip_conv2d_pointwise_block_weight_bytes)
STUB_UNUSED(avhip_conv2d_pointwise_block_weight_layout)
STUB_UNUSED(avhip_conv2d_winograd_rows)
STUB_UNUSED(avhip_im2row)
STUB_UNUSED(avhip_set_conv_strided)
STUB_UNUSED(avhip_set_memory)
STUB_UNUSED(avhip_set_pointwise_block)
STUB_UNUSED(avhip_set_winograd_rows)
STUB_UNUSED(avhip_winograd_gradient_transform)
STUB_UNUSED(avhip_winograd_rows_weight_bytes)
STUB_UNUSED(avhip_winograd_rows_weight_transform)
STUB_UNUSED(avhip_winograd_update_transform)

namespace avhip
{
	bool winograd_f4_takes(const avhipConvShape&, const void*, const void*, const void*, double, int activation)
	{
		return activation == 0 || activation == 3;
	}
}

"""Tensors beyond 2 GiB: the kernels' 32-bit-offset fast paths must hand such problems to the instances with 64-bit indexing.
Every image of a batch is independent, so images are generated, uploaded and checked one at a time against the CPU oracle:
the first, a middle and the last image (whose bytes lie beyond the 2 GiB mark) through the C API."""
import ctypes as C

import numpy as np
import pytest

import cudabackend_amd as cb
import helpers as h

pytestmark = pytest.mark.gpu


def image(seed, shape, kind):
    g = np.random.default_rng(1000 + seed)
    if kind == "i8":
        return g.integers(-127, 128, shape, dtype=np.int8)
    return g.standard_normal(shape, dtype=np.float32).astype(np.float16)


def upload_images(lib, ctx, tensor, n_images, shape, kind):
    per = int(np.prod(shape)) * (1 if kind == "i8" else 2)
    for i in range(n_images):
        raw = np.ascontiguousarray(image(i, shape, kind))
        cb.check(lib.cudaCopyMemoryFromHost(ctx, tensor.mem, i * per, raw.ctypes.data_as(C.c_void_p), per), "upload")


def download_image(lib, ctx, tensor, index, shape, np_dtype):
    out = np.empty(shape, dtype=np_dtype)
    cb.check(lib.cudaCopyMemoryToHost(ctx, out.ctypes.data_as(C.c_void_p), tensor.mem, index * out.nbytes, out.nbytes), "download")
    return out


def test_int8_pointwise_beyond_2gib_bit_exact(oracle):
    N, H, W, Cin, K = 36, 1024, 1024, 64, 16          # x 2.42 GB int8, y 2.42 GB int32
    lib = cb.load_library()
    ctx = lib.cudaGetDefaultContext(0)
    g = h.rng(70)
    w = g.integers(-127, 128, (K, 1, 1, Cin), dtype=np.int8)
    b = g.integers(-2 ** 15, 2 ** 15, K).astype(np.int32)
    x = cb.DeviceTensor((N, H, W, Cin), cb.DTYPE_INT8, zero=False)
    y = cb.DeviceTensor((N, H, W, K), cb.DTYPE_INT32, zero=False)
    assert x.nbytes > 2 ** 31 and y.nbytes > 2 ** 31
    wt, bt = cb.DeviceTensor.from_numpy(w, cb.DTYPE_INT8), cb.DeviceTensor.from_numpy(b, cb.DTYPE_INT32)
    upload_images(lib, ctx, x, N, (H, W, Cin), "i8")
    conv = cb.ConvolutionDescriptor(padding=(0, 0), dtype=cb.DTYPE_INT8)
    print("int8 1x1 beyond 2 GiB", flush=True)
    cb.check(lib.cudaConvolutionImplicitGemmForward(ctx, conv.handle, None, x.desc, x.mem, wt.desc, wt.mem, bt.desc, bt.mem, None, 0, 0, None,
                                                     y.desc, y.mem, cb.ACTIVATION_RELU), "conv")
    cb.check(lib.cudaSynchronizeWithContext(ctx), "sync")
    for i in (0, N // 2, N - 1):
        got = download_image(lib, ctx, y, i, (H, W, K), np.int32)
        want = oracle.conv2d_i8(image(i, (1, H, W, Cin), "i8"), w, b, pad=(0, 0), activation=oracle.RELU)[0]
        np.testing.assert_array_equal(got, want)
    for t in (x, y, wt, bt):
        t.close()


def test_fp16_3x3_beyond_2gib(oracle):
    N, H, W, Cin, K = 9, 2048, 2048, 32, 8            # x 2.42 GB fp16
    lib = cb.load_library()
    ctx = lib.cudaGetDefaultContext(0)
    g = h.rng(71)
    w = h.rounded(oracle, g.standard_normal((K, 3, 3, Cin)) * np.sqrt(2.0 / (9 * Cin)), "f16")
    b = g.uniform(-0.1, 0.1, K).astype(np.float32).astype(np.float64)
    x = cb.DeviceTensor((N, H, W, Cin), cb.DTYPE_FLOAT16, zero=False)
    y = cb.DeviceTensor((N, H, W, K), cb.DTYPE_FLOAT16, zero=False)
    assert x.nbytes > 2 ** 31
    wt, bt = cb.DeviceTensor.from_numpy(w, cb.DTYPE_FLOAT16), cb.DeviceTensor.from_numpy(b, cb.DTYPE_FLOAT32)
    upload_images(lib, ctx, x, N, (H, W, Cin), "f16")
    conv = cb.ConvolutionDescriptor(padding=(-1, -1), dtype=cb.DTYPE_FLOAT16)
    print("fp16 3x3 beyond 2 GiB", flush=True)
    cb.check(lib.cudaConvolutionImplicitGemmForward(ctx, conv.handle, None, x.desc, x.mem, wt.desc, wt.mem, bt.desc, bt.mem, None, 0, 0, None,
                                                     y.desc, y.mem, cb.ACTIVATION_RELU), "conv")
    cb.check(lib.cudaSynchronizeWithContext(ctx), "sync")
    for i in (0, N - 1):
        got = download_image(lib, ctx, y, i, (H, W, K), np.float16).astype(np.float64)
        want = oracle.conv2d(image(i, (1, H, W, Cin), "f16").astype(np.float64), w, b, activation=oracle.RELU)[0]
        err = oracle.rel_l2(got, want)
        print("image %d rel-L2 = %.3e" % (i, err))
        assert err < 2e-3
    for t in (x, y, wt, bt):
        t.close()


def test_tn_product_of_more_tiles_than_one_launch_takes():
    """65535 products 1 x 8193 over k = 1: 257 tiles of 32 columns (129 of 64) each are 16.8 (8.5) million workgroups of 512 work-items,
    beyond the 2^32 work-items of one launch; the generic kernel, whose grid has three directions, has to take them.  One product per
    output, rounded once: exact."""
    batch, N, chunk = 65535, 8193, 4369
    lib = cb.load_library()
    ctx = lib.cudaGetDefaultContext(0)
    a = ((np.arange(batch) % 61) * 0.25 - 7).astype(np.float16)
    row = np.random.default_rng(14).standard_normal(N).astype(np.float16)
    A = cb.DeviceTensor((batch, 1, 1), cb.DTYPE_FLOAT16, zero=False)
    B, Y = (cb.DeviceTensor((batch, 1, N), cb.DTYPE_FLOAT16, zero=False) for _ in range(2))
    cb.check(lib.cudaCopyMemoryFromHost(ctx, A.mem, 0, a.ctypes.data_as(C.c_void_p), a.nbytes), "upload")
    rows = np.ascontiguousarray(np.broadcast_to(row, (chunk, N)))
    for i in range(0, batch, chunk):
        cb.check(lib.cudaCopyMemoryFromHost(ctx, B.mem, i * row.nbytes, rows.ctypes.data_as(C.c_void_p), rows.nbytes), "upload")
    print("fp16 (T, N) product, 65535 x 1 x 8193", flush=True)
    cb.check(lib.cudaGemmBatched(ctx, cb.GEMM_OPERATION_T, cb.GEMM_OPERATION_N, None, A.desc, A.mem, B.desc, B.mem, None, Y.desc, Y.mem), "cudaGemmBatched")
    cb.check(lib.cudaSynchronizeWithContext(ctx), "sync")
    for i in (0, 1, batch // 2, batch - 1):
        want = (a[i].astype(np.float32) * row.astype(np.float32)).astype(np.float16)
        np.testing.assert_array_equal(download_image(lib, ctx, Y, i, (N,), np.float16), want)
    for t in (A, B, Y):
        t.close()


def test_more_output_pixels_than_small_tiles_take_in_one_launch():
    """540 million output pixels, all but four of them border: 16.9 million tiles of 32 pixels with four wavefronts each would be more
    than 2^32 work-items.  The layer (1929 channels: no whole number of 16-byte chunks) has to be left to the gather kernel."""
    lib = cb.load_library()
    ctx = lib.cudaGetDefaultContext(0)
    offset, Cin, K = 23240, 1929, 4
    side = 2 + offset
    assert (side * side + 31) // 32 * 256 >= 1 << 32
    g = h.rng(71)
    x, w = (g.standard_normal(s).astype(np.float16) for s in ((1, 2, 2, Cin), (K, 1, 1, Cin)))
    xt, wt = cb.DeviceTensor.from_numpy(x, cb.DTYPE_FLOAT16), cb.DeviceTensor.from_numpy(w, cb.DTYPE_FLOAT16)
    bias = np.array([0.5, -1.0, 2.0, 0.25])
    bt = cb.DeviceTensor.from_numpy(bias, cb.DTYPE_FLOAT32)
    y = cb.DeviceTensor((1, side, side, K), cb.DTYPE_FLOAT16)
    conv = cb.ConvolutionDescriptor(padding=(-offset, -offset), dtype=cb.DTYPE_FLOAT16)
    print("fp16 1x1 with 23240 rows and columns of border", flush=True)
    cb.check(lib.cudaConvolutionImplicitGemmForward(ctx, conv.handle, None, xt.desc, xt.mem, wt.desc, wt.mem, bt.desc, bt.mem, None, 0, 0, None,
                                                     y.desc, y.mem, cb.ACTIVATION_LINEAR), "conv")
    cb.check(lib.cudaSynchronizeWithContext(ctx), "sync")
    for row in (0, 1, side // 3, offset - 1, offset, offset + 1):
        got = download_image(lib, ctx, y, row, (side, K), np.float16).astype(np.float64)
        want = np.broadcast_to(bias, (side, K)).copy()
        if offset <= row < offset + 2:
            want[offset:offset + 2] += x[0, row - offset].astype(np.float64) @ w[:, 0, 0].astype(np.float64).T
        np.testing.assert_allclose(got, want, rtol=2e-3, atol=2e-2)  # a sum of 1929 products of size 1 in fp32, rounded to fp16
    for t in (xt, wt, bt, y):
        t.close()

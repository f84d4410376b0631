"""Which tiles the A^T B product of the weight gradient takes in fp32 (csrc/gemm_tn.hip): products of the shapes of Winograd gradients, each timed with both,
go to the faster one.  Host arithmetic only."""
import pytest

import cudabackend_amd as cb

# batch, M, N, K; microseconds in tiles of 32 (fp32 products) and of 64 (bf16 pieces)
TIMED = [((36, 80, 224, 2150), 36.6, 54.7), ((36, 96, 208, 2793), 43.8, 65.2), ((36, 216, 32, 1716), 15.5, 22.7), ((36, 32, 208, 203), 5.7, 7.3),
         ((36, 216, 128, 441), 14.5, 18.4), ((36, 112, 216, 2489), 51.8, 61.5), ((36, 88, 216, 531), 17.2, 19.7), ((36, 48, 200, 464), 8.6, 9.7),
         ((36, 128, 128, 512), 11.4, 9.7), ((36, 168, 128, 273), 14.1, 8.5), ((36, 104, 168, 113), 14.1, 7.6), ((36, 168, 256, 735), 38.6, 26.1),
         ((16, 224, 224, 2162), 45.5, 31.5), ((36, 240, 240, 2324), 103.7, 89.6), ((16, 248, 192, 2983), 42.9, 35.5), ((36, 248, 224, 147), 26.7, 19.7),
         ((16, 96, 40, 1460), 9.3, 18.5), ((36, 64, 64, 1666), 11.7, 21.4), ((16, 104, 192, 7128), 58.5, 69.3)]


@pytest.mark.parametrize("shape, small, large", TIMED)
def test_the_faster_tiles_are_taken(shape, small, large):
    assert cb.load_library().avhip_gemm_tn_side(4, *shape) == (64 if large < small else 32)


@pytest.mark.parametrize("batch", [2 ** 15, 2 ** 20, 2 ** 23, 2 ** 31 - 1])
def test_no_more_work_items_than_a_launch_takes(batch):
    """A product of one tile of either size: small ones until they are 2^32 work-items."""
    side = cb.load_library().avhip_gemm_tn_side(4, batch, 32, 64, 16)
    assert side == 64 if 2 * batch * 512 >= 2 ** 32 else side == 32

"""The dispatcher's choice among the one-kernel plans, held against the clock on the layers of the BASELINE configurations: the plan
it takes by itself must not be slower than what it would run with that plan switched off.  (Parity of every plan is tested
elsewhere; this pins that the thresholds of `rows_winograd_pays`, `strided_kernel_pays` and `pointwise_block_pays` point the
right way where it matters.)  Times are HIP events around graph replays, the same helper bench.py uses; the margin of 10 % is far
inside the differences measured (30-55 %), so the box-to-box spread of the clocks does not decide the outcome."""
import pytest

import cudabackend_amd as cb

pytestmark = pytest.mark.gpu

# name, dtype, x, w, padding, stride; the switch of the plan the dispatcher is expected to take
LAYERS = [
    (("config 2 body 3x3 128->128", "bf16", (256, 15, 15, 128), (128, 3, 3, 128), -1, 1), "avhip_set_winograd_rows"),
    (("config 3 3x3 256->256", "bf16", (64, 56, 56, 256), (256, 3, 3, 256), -1, 1), "avhip_set_winograd_rows"),
    (("config 5 3x3 stride 2 128->256", "bf16", (64, 56, 56, 128), (256, 3, 3, 128), -1, 2), "avhip_set_conv_strided"),
    (("config 5 1x1 256->512", "bf16", (64, 28, 28, 256), (512, 1, 1, 256), 0, 1), "avhip_set_pointwise_block"),
]


@pytest.mark.parametrize("case", range(len(LAYERS)))
def test_the_plan_taken_is_not_the_slower_one(case):
    import bench
    layer, switch = LAYERS[case]
    lib = cb.load_library()
    setter = getattr(lib, switch)
    setter.restype = int
    hip, ctx = bench.Hip(), cb.Context(0)
    times = {}
    previous = setter(1)
    try:
        for mode in (1, 0, 1, 0):
            setter(mode)
            us = bench.other_configs(hip, ctx, 10, [layer])[layer[0]]["us"]
            times[mode] = min(times.get(mode, us), us)
    finally:
        setter(previous)
        ctx.close()
    print("%s: %.1f us with the plan, %.1f us without" % (layer[0], times[1], times[0]))
    assert times[1] <= 1.10 * times[0]


# layers at which the estimates of the kernel of small tiles have to point the right way: name, dtype, x, w, padding, stride
SMALL_OR_NOT = [
    ("1x1 16->12, which the one-tap kernels decline", "bf16", (40, 12, 12, 16), (12, 1, 1, 16), 0, 1),
    ("1x1 96->44, likewise", "f16", (7, 20, 20, 96), (44, 1, 1, 96), 0, 1),
    ("1x1 116->44 in fp32: a chain of four steps in the one-tap kernels", "f32", (3, 12, 12, 116), (44, 1, 1, 116), 0, 1),
    ("1x1 256->512: the one-tap kernels'", "bf16", (16, 28, 28, 256), (512, 1, 1, 256), 0, 1),
    ("3x3 28->196, packed gather", "bf16", (52, 56, 56, 28), (196, 3, 3, 28), -1, 1),
    ("3x3 6->100 on few pixels, not the packed gather", "f16", (4, 28, 28, 6), (100, 3, 3, 6), -1, 1),
    ("3x3 484->92 on few pixels, offered a split of k", "f32", (1, 16, 16, 484), (92, 3, 3, 484), -1, 1),
    ("3x3 128->128, four workgroups more than a round", "f16", (129, 18, 18, 128), (128, 3, 3, 128), -1, 1),
    ("3x3 64->64 on few pixels", "f32", (8, 15, 15, 64), (64, 3, 3, 64), -1, 1),
]


@pytest.mark.parametrize("case", range(len(SMALL_OR_NOT)))
def test_small_tiles_are_taken_where_they_are_the_faster_ones(case):
    """Threshold of the kernel of small tiles: default, never, always.  The default must not be slower than either by more than a
    quarter (but for the layer of one round and a bit, where that is the whole difference: a tenth): the differences it has to tell apart
    here are factors of 1.15 to 2.5, and its estimates are off by 6 to 13 %."""
    import bench
    layer = SMALL_OR_NOT[case]
    lib = cb.load_library()
    lib.avhip_set_small_problem_threshold.restype = int
    hip, ctx = bench.Hip(), cb.Context(0)
    times = {}
    previous = lib.avhip_set_small_problem_threshold(4096)
    try:
        for mode in (4096, 0, -1, 4096, 0, -1):
            lib.avhip_set_small_problem_threshold(mode)
            us = bench.other_configs(hip, ctx, 20, [layer])[layer[0]]["us"]
            times[mode] = min(times.get(mode, us), us)
    finally:
        lib.avhip_set_small_problem_threshold(previous)
        ctx.close()
    print("%s: %.1f us, without small tiles %.1f, with %.1f" % (layer[0], times[4096], times[0], times[-1]))
    assert times[4096] <= (1.1 if "more than a round" in layer[0] else 1.25) * min(times[0], times[-1])

"""What a program built on this backend spends its time in, as cases that can be timed and compared: convolution layers of all
kinds through the dispatcher, residual towers from one position to a full batch, the quantised pair of layers, the non-fused
Winograd stages called one by one, and the Winograd weight gradient of a training step.  Everything goes through the C API of
include/avocado_hip_backend.h as cudabackend_amd.api binds it; PyTorch only makes the inputs and looks at the outputs.
"""
import ctypes as C
import math

import torch  # before the backend, so that both use one HIP runtime

import cudabackend_amd as cb

DTYPE = {"f32": cb.DTYPE_FLOAT32, "f16": cb.DTYPE_FLOAT16, "bf16": cb.DTYPE_BFLOAT16, "i8": cb.DTYPE_INT8, "i32": cb.DTYPE_INT32, "u8": cb.DTYPE_UINT8}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8, "i32": torch.int32, "u8": torch.uint8}
SIZE = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1, "i32": 4, "u8": 1}
TYPESTR = {1: "|u1", 2: "<i2", 4: "<i4"}
ACTIVATION = {"linear": cb.ACTIVATION_LINEAR, "relu": cb.ACTIVATION_RELU, "sigmoid": cb.ACTIVATION_SIGMOID, "tanh": cb.ACTIVATION_TANH,
              "elu": cb.ACTIVATION_ELU}


def listed():
    return [
        # one small fp32 layer of a batch of eight positions; launch and host latency count
        {"name": "layer_small_f32", "kind": "layer", "dtype": "f32", "n": 8, "h": 15, "w": 15, "c": 64, "k": 64, "r": 3, "stride": 1, "residual": False,
         "act": "relu"},
        # one position evaluated alone, as a player or a search without batching does: 21 dependent calls
        {"name": "tower_one_f16", "kind": "tower", "dtype": "f16", "n": 1, "size": 15, "ch": 128, "blocks": 10},
        # BASELINE config 2, the headline: a full batch of 256 positions through ten residual blocks
        {"name": "tower_bf16", "kind": "tower", "dtype": "bf16", "n": 256, "size": 15, "ch": 128, "blocks": 10},
        # the same in fp32, where the Winograd plans with a workspace run
        {"name": "tower_f32", "kind": "tower", "dtype": "f32", "n": 256, "size": 15, "ch": 128, "blocks": 10},
        # the large layer of an image network
        {"name": "layer_large_bf16", "kind": "layer", "dtype": "bf16", "n": 64, "h": 56, "w": 56, "c": 256, "k": 256, "r": 3, "stride": 1,
         "residual": False, "act": "relu"},
        # a downsampling layer and the 1x1 layer that widens its output
        {"name": "downsample_bf16", "kind": "downsample", "dtype": "bf16", "n": 64, "h": 56, "w": 56, "c": 128},
        # the 5x5 layer
        {"name": "layer_5x5_bf16", "kind": "layer", "dtype": "bf16", "n": 64, "h": 32, "w": 32, "c": 64, "k": 64, "r": 5, "stride": 1,
         "residual": False, "act": "relu"},
        # sizes that divide by nothing in particular: a narrow network on a larger board, with a residual
        {"name": "layer_ragged_f16", "kind": "layer", "dtype": "f16", "n": 37, "h": 19, "w": 17, "c": 72, "k": 100, "r": 3, "stride": 1,
         "residual": True, "act": "elu"},
        # the first layer of an image network: three planes
        {"name": "layer_first_bf16", "kind": "layer", "dtype": "bf16", "n": 32, "h": 224, "w": 224, "c": 3, "k": 64, "r": 7, "stride": 2,
         "residual": False, "act": "relu"},
        # BASELINE config 4 as a network runs it: 3x3 requantised to int8, its output through 1x1 to int32
        {"name": "quantised_i8", "kind": "quantised", "n": 128, "h": 20, "w": 20, "c": 128, "k": 128},
        # the non-fused Winograd stages one by one, as a front-end that keeps its own transformed weights calls them (config 2 layer)
        {"name": "stages_bf16", "kind": "stages", "dtype": "bf16", "m": 2, "n": 256, "h": 15, "w": 15, "c": 128, "k": 128},
        # training: the weight gradient of a config 2 layer at a training batch, through the Winograd domain
        {"name": "weight_gradient_f32", "kind": "weight_gradient", "dtype": "f32", "m": 4, "n": 32, "h": 15, "w": 15, "c": 128, "k": 128},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _channels(rng, low, high):
    """Mostly multiples of 8 or of 32, now and then any number."""
    v, kind = _log(rng, low, high), rng.random()
    if kind < 0.45:
        return max(32, 32 * round(v / 32))
    return max(8, 8 * round(v / 8)) if kind < 0.85 else v


def draw(rng):
    """One more case of the ranges above, none dearer than the dearest of them."""
    kind = rng.choices(["layer", "first", "tower", "downsample", "quantised", "stages", "weight_gradient"], [8, 2, 3, 1.5, 2, 1.5, 2])[0]
    while True:
        if kind == "layer":
            h = _log(rng, 7, 64)
            case = {"kind": "layer", "dtype": rng.choice(["f32", "f16", "bf16"]), "n": _log(rng, 1, 256), "h": h, "w": max(7, h + rng.choice([0, 0, -1, 1, 3, -4])),
                    "c": _channels(rng, 16, 512), "k": _channels(rng, 16, 512), "r": rng.choice([1, 3, 3, 3, 5]), "stride": rng.choice([1, 1, 1, 2]),
                    "residual": rng.random() < 0.35, "act": rng.choice(["relu", "relu", "relu", "linear", "sigmoid", "tanh", "elu"])}
        elif kind == "first":
            h = _log(rng, 15, 224)
            case = {"kind": "layer", "dtype": rng.choice(["f32", "f16", "bf16"]), "n": _log(rng, 1, 64), "h": h, "w": h + rng.choice([0, 0, -1, 5]),
                    "c": rng.choice([1, 2, 3, 3, 4, 8]), "k": 16 * rng.randint(2, 8), "r": rng.choice([3, 5, 7]), "stride": rng.choice([1, 2]),
                    "residual": False, "act": rng.choice(["relu", "linear"])}
        elif kind == "tower":
            case = {"kind": "tower", "dtype": rng.choice(["f32", "f16", "bf16"]), "n": _log(rng, 1, 256), "size": rng.randint(9, 20),
                    "ch": rng.choice([32, 64, 96, 128, 128, 192, 256]), "blocks": rng.randint(2, 10)}
        elif kind == "downsample":
            h = _log(rng, 14, 64)
            case = {"kind": "downsample", "dtype": rng.choice(["f16", "bf16"]), "n": _log(rng, 4, 128), "h": h, "w": h + rng.choice([0, 0, -1, 3]),
                    "c": 32 * rng.randint(1, 8)}
        elif kind == "quantised":
            h = _log(rng, 8, 48)
            case = {"kind": "quantised", "n": _log(rng, 1, 256), "h": h, "w": h + rng.choice([0, 0, -1, 3]), "c": 16 * rng.randint(2, 16),
                    "k": 16 * rng.randint(2, 16)}
        else:
            dtype = rng.choice(["f32", "f16", "bf16"])
            h = _log(rng, 9, 40)
            case = {"kind": kind, "dtype": dtype, "m": rng.choice([2, 4]) if dtype == "f32" else 2,
                    "n": _log(rng, 4, 256) if kind == "stages" else _log(rng, 4, 64), "h": h, "w": h + rng.choice([0, 0, -1, 3]),
                    "c": _channels(rng, 32, 256), "k": _channels(rng, 32, 256)}
        need = work(case)
        most = 60e9 if case["kind"] != "tower" else 200e9
        if need["flops"] <= (most if case.get("dtype") != "f32" else most / 3) and need["bytes"] <= 400e6:
            return case


# ---- device memory of the backend, seen as torch tensors ---------------------------------------------------------------------------
class _Address:
    """Hands torch the address of a tensor of the backend (and keeps the tensor while torch holds the view)."""

    def __init__(self, tensor, item):
        self.tensor = tensor
        self.__cuda_array_interface__ = {"shape": tensor.shape, "typestr": TYPESTR[item], "data": (tensor.pointer(), False), "version": 2, "strides": None}


def _view(tensor, dtype):
    return torch.as_tensor(_Address(tensor, SIZE[dtype]), device="cuda").view(TORCH[dtype])


class _Made:
    """Tensors of the backend filled from one seed."""

    def __init__(self, seed):
        self.random = torch.Generator(device="cuda")
        self.random.manual_seed(seed)
        self.lib = cb.load_library()

    def empty(self, shape, dtype):
        return cb.DeviceTensor(shape, DTYPE[dtype], zero=False)

    def filled(self, values, dtype):
        t = self.empty(tuple(values.shape), dtype)
        _view(t, dtype).copy_(values)
        return t

    def normal(self, shape, dtype, scale=1.0):
        return self.filled(torch.randn(shape, generator=self.random, device="cuda") * scale, dtype)

    def uniform(self, shape, dtype, low, high):
        return self.filled(torch.rand(shape, generator=self.random, device="cuda") * (high - low) + low, dtype)

    def planes(self, shape, dtype):
        """Board planes: about 15 of 100 points set."""
        return self.filled((torch.rand(shape, generator=self.random, device="cuda") < 0.15).float(), dtype)

    def integers(self, shape, dtype, low, high):
        return self.filled(torch.randint(low, high, shape, generator=self.random, device="cuda"), dtype)

    def weights(self, k, r, c, dtype):
        return self.normal((k, r, r, c), dtype, math.sqrt(2.0 / (r * r * c)))


_the_context = []


def _context():
    """The one context (one stream) such a program works on."""
    if not _the_context:
        _the_context.append(cb.Context(0))
    return _the_context[0]


def _out(size, r, stride):
    return (size + 2 * (r // 2) - r) // stride + 1


class _Layer:
    """One call of the dispatcher with everything it needs in hand."""

    def __init__(self, made, dtype, x, w, b, z, y, stride, act, workspace=None):
        self.x, self.w, self.b, self.z, self.y, self.act = x, w, b, z, y, ACTIVATION[act]
        pad = -(w.shape[1] // 2)
        self.conv = cb.ConvolutionDescriptor(padding=(pad, pad), strides=(stride, stride), dtype=DTYPE[dtype])
        self.lib, self.context = made.lib, _context()
        need = C.c_int64(0)
        cb.check(self.lib.cudaGetConvolutionWorkspaceSize(self.context.handle, self.conv.handle, x.desc, w.desc, b.desc, C.byref(need)),
                 "cudaGetConvolutionWorkspaceSize")
        self.workspace = workspace
        if need.value and (workspace is None or workspace.nbytes < need.value):
            self.workspace = made.empty((need.value,), "u8")

    def forward(self):
        x, w, b, z, y = self.x, self.w, self.b, self.z, self.y
        cb.check(self.lib.cudaConvolutionBiasActivationForward(
            self.context.handle, self.conv.handle, None, x.desc, x.mem, w.desc, w.mem, b.desc, b.mem, None, z.desc if z is not None else 0,
            z.mem if z is not None else 0, None, y.desc, y.mem, self.act, self.workspace.mem if self.workspace is not None else 0),
            "cudaConvolutionBiasActivationForward")


class _Stages:
    """The Winograd entry points called one by one."""

    def __init__(self, case, made):
        dtype, m = case["dtype"], case["m"]
        n, h, w, c, k = (case[key] for key in ("n", "h", "w", "c", "k"))
        matrices = "f32" if dtype == "f32" else "f16"
        t, tiles = m + 2, n * -(-h // m) * -(-w // m)
        self.m, self.lib, self.context = m, made.lib, _context()
        self.conv = cb.ConvolutionDescriptor(padding=(-1, -1), dtype=DTYPE[dtype])
        self.x = made.normal((n, h, w, c), dtype)
        self.weight = made.weights(k, 3, c, dtype)
        self.V = made.empty((t * t, tiles, c), matrices)
        if case["kind"] == "stages":
            self.bias = made.uniform((k,), "f32", -0.1, 0.1)
            self.U = made.empty((t * t, k, c), matrices)
            self.M = made.empty((t * t, tiles, k), "f32")
            self.y = made.empty((n, h, w, k), dtype)
            torch.cuda.synchronize()
            cb.check(self.lib.cudaWinogradWeightTransform(self.context.handle, self.conv.handle, m, self.weight.desc, self.weight.mem, self.U.desc,
                                                          self.U.mem), "cudaWinogradWeightTransform")
            self.out = _view(self.y, dtype)
        else:
            self.dy = made.normal((n, h, w, k), dtype, 0.05)
            self.G = made.empty((t * t, tiles, k), matrices)
            self.P = made.empty((t * t, k, c), "f32")
            self.dw = made.empty((k, 3, 3, c), dtype)
            self.out = _view(self.dw, dtype)

    def input_transform(self):
        cb.check(self.lib.cudaWinogradInputTransform(self.context.handle, self.conv.handle, self.m, self.weight.desc, self.x.desc, self.x.mem, self.V.desc,
                                                     self.V.mem), "cudaWinogradInputTransform")

    def forward(self):
        handle, conv, m = self.context.handle, self.conv.handle, self.m
        self.input_transform()
        cb.check(self.lib.cudaGemmBatched(handle, cb.GEMM_OPERATION_N, cb.GEMM_OPERATION_T, None, self.V.desc, self.V.mem, self.U.desc, self.U.mem, None,
                                          self.M.desc, self.M.mem), "cudaGemmBatched")
        cb.check(self.lib.cudaWinogradOutputTransform(handle, conv, m, self.weight.desc, None, self.M.desc, self.M.mem, self.y.desc, self.y.mem,
                                                      self.bias.desc, self.bias.mem, None, 0, 0, None, cb.ACTIVATION_RELU), "cudaWinogradOutputTransform")
        return self.out

    def weight_gradient(self):
        handle, conv, m = self.context.handle, self.conv.handle, self.m
        self.input_transform()
        cb.check(self.lib.cudaWinogradGradientTransform(handle, conv, m, self.weight.desc, self.dy.desc, self.dy.mem, self.G.desc, self.G.mem),
                 "cudaWinogradGradientTransform")
        cb.check(self.lib.cudaGemmBatched(handle, cb.GEMM_OPERATION_T, cb.GEMM_OPERATION_N, None, self.G.desc, self.G.mem, self.V.desc, self.V.mem, None,
                                          self.P.desc, self.P.mem), "cudaGemmBatched")
        cb.check(self.lib.cudaWinogradUpdateTransform(handle, conv, m, None, self.P.desc, self.P.mem, None, self.dw.desc, self.dw.mem),
                 "cudaWinogradUpdateTransform")
        return self.out


def prepare(case, seed):
    made, kind = _Made(seed), case["kind"]
    if kind == "layer":
        dtype, n, h, w, c, k, r, stride = (case[key] for key in ("dtype", "n", "h", "w", "c", "k", "r", "stride"))
        x = made.normal((n, h, w, c), dtype)
        shape = (n, _out(h, r, stride), _out(w, r, stride), k)
        z = made.normal(shape, dtype) if case["residual"] else None
        y = made.empty(shape, dtype)
        layers = [_Layer(made, dtype, x, made.weights(k, r, c, dtype), made.uniform((k,), "f32", -0.1, 0.1), z, y, stride, case["act"])]
        state = {"layers": layers, "out": _view(y, dtype)}
    elif kind == "tower":
        dtype, n, size, ch = (case[key] for key in ("dtype", "n", "size", "ch"))
        a, t, b = (made.empty((n, size, size, ch), dtype) for _ in range(3))
        layers = [_Layer(made, dtype, made.planes((n, size, size, 4), dtype), made.weights(ch, 3, 4, dtype), made.uniform((ch,), "f32", -0.1, 0.1), None, a,
                         1, "relu")]
        workspace = None
        for _ in range(case["blocks"]):
            for x, z, y in ((a, None, t), (t, a, b)):
                layers.append(_Layer(made, dtype, x, made.weights(ch, 3, ch, dtype), made.uniform((ch,), "f32", -0.1, 0.1), z, y, 1, "relu", workspace))
                workspace = layers[-1].workspace
            a, b = b, a
        state = {"layers": layers, "out": _view(a, dtype)}
    elif kind == "downsample":
        dtype, n, h, w, c = (case[key] for key in ("dtype", "n", "h", "w", "c"))
        ho, wo = _out(h, 3, 2), _out(w, 3, 2)
        x, y, v = made.normal((n, h, w, c), dtype), made.empty((n, ho, wo, 2 * c), dtype), made.empty((n, ho, wo, 4 * c), dtype)
        layers = [_Layer(made, dtype, x, made.weights(2 * c, 3, c, dtype), made.uniform((2 * c,), "f32", -0.1, 0.1), None, y, 2, "relu"),
                  _Layer(made, dtype, y, made.weights(4 * c, 1, 2 * c, dtype), made.uniform((4 * c,), "f32", -0.1, 0.1), None, v, 1, "relu")]
        state = {"layers": layers, "out": (_view(y, dtype), _view(v, dtype))}
    elif kind == "quantised":
        n, h, w, c, k = (case[key] for key in ("n", "h", "w", "c", "k"))
        state = {"lib": made.lib, "context": _context(), "x": made.integers((n, h, w, c), "i8", -127, 128),
                 "w3": made.integers((k, 3, 3, c), "i8", -127, 128), "w1": made.integers((k, 1, 1, k), "i8", -127, 128),
                 "b3": made.integers((k,), "i32", -2 ** 15, 2 ** 15), "b1": made.integers((k,), "i32", -2 ** 15, 2 ** 15),
                 "scale": made.uniform((k,), "f32", 1e-4, 1e-3), "q": made.empty((n, h, w, k), "i8"), "y": made.empty((n, h, w, k), "i32"),
                 "conv3": cb.ConvolutionDescriptor(padding=(-1, -1), dtype=cb.DTYPE_INT8), "conv1": cb.ConvolutionDescriptor(padding=(0, 0), dtype=cb.DTYPE_INT8)}
        state["out"] = (_view(state["q"], "i8"), _view(state["y"], "i32"))
    else:
        state = {"stages": _Stages(case, made)}
    state["kind"] = kind
    torch.cuda.synchronize()
    return state


def run(state):
    if state["kind"] == "stages":
        return state["stages"].forward()
    if state["kind"] == "weight_gradient":
        return state["stages"].weight_gradient()
    if state["kind"] == "quantised":
        lib, handle, x, q, y, w3, w1, b3, b1, scale = (state[key] for key in ("lib", "context", "x", "q", "y", "w3", "w1", "b3", "b1", "scale"))
        handle = handle.handle
        cb.check(lib.avhipConvolutionRequantForward(handle, state["conv3"].handle, x.desc, x.mem, w3.desc, w3.mem, b3.desc, b3.mem, scale.desc, scale.mem,
                                                    q.desc, q.mem, cb.ACTIVATION_RELU), "avhipConvolutionRequantForward")
        cb.check(lib.cudaConvolutionImplicitGemmForward(handle, state["conv1"].handle, None, q.desc, q.mem, w1.desc, w1.mem, b1.desc, b1.mem, None, 0, 0,
                                                        None, y.desc, y.mem, cb.ACTIVATION_LINEAR), "cudaConvolutionImplicitGemmForward")
        return state["out"]
    for layer in state["layers"]:
        layer.forward()
    return state["out"]


def _conv_work(size, n, h, w, c, k, r, stride=1, residual=False, out_size=None):
    pixels = n * _out(h, r, stride) * _out(w, r, stride)
    out_size = out_size or size
    return {"bytes": size * (n * h * w * c + k * r * r * c) + out_size * pixels * k * (2 if residual else 1) + 4 * k, "flops": 2.0 * pixels * k * r * r * c}


def work(case):
    """Convolutions are counted as the direct form's operations.  The stages called one by one hand V, M (and the gradient's
    matrices) to each other through memory: each is written once and read once."""
    kind = case["kind"]
    if kind == "layer":
        parts = [_conv_work(SIZE[case["dtype"]], case["n"], case["h"], case["w"], case["c"], case["k"], case["r"], case["stride"], case["residual"])]
    elif kind == "tower":
        size, args = SIZE[case["dtype"]], (case["n"], case["size"], case["size"])
        parts = [_conv_work(size, *args, 4, case["ch"], 3)]
        parts += case["blocks"] * [_conv_work(size, *args, case["ch"], case["ch"], 3, residual=z) for z in (False, True)]
    elif kind == "downsample":
        n, h, w, c = (case[key] for key in ("n", "h", "w", "c"))
        parts = [_conv_work(2, n, h, w, c, 2 * c, 3, 2), _conv_work(2, n, _out(h, 3, 2), _out(w, 3, 2), 2 * c, 4 * c, 1)]
    elif kind == "quantised":
        n, h, w, c, k = (case[key] for key in ("n", "h", "w", "c", "k"))
        parts = [_conv_work(1, n, h, w, c, k, 3), _conv_work(1, n, h, w, k, k, 1, out_size=4)]
    else:
        n, h, w, c, k, m = (case[key] for key in ("n", "h", "w", "c", "k", "m"))
        size = SIZE[case["dtype"]]
        matrix, points, tiles = (4 if size == 4 else 2), (m + 2) ** 2, n * -(-h // m) * -(-w // m)
        flops, x, y = 2.0 * points * tiles * c * k, size * n * h * w * c, size * n * h * w * k
        if kind == "stages":
            total = x + y + 4 * k + matrix * points * (2 * tiles * c + k * c) + 2 * 4 * points * tiles * k
        else:
            total = x + y + size * k * 9 * c + matrix * points * 2 * tiles * (c + k) + 2 * 4 * points * k * c
        parts = [{"bytes": total, "flops": flops}]
    return {key: float(sum(p[key] for p in parts)) for key in ("bytes", "flops")}


def tolerance(case):
    """About four times the largest relative error (2-norm) seen against the same pass in 64 bits, the chains with every layer's
    output rounded to its type: 32-bit 0.3e-6 .. 1e-6 for a layer (direct and Winograd plans), 2e-6 for a tower, 2.5e-6 for the
    F(4x4, 3x3) stages, 9e-6 for their weight gradient; fp16 3.5e-4, 8e-4 and 5.3e-4; bf16 1.7e-3 (the last rounding) and 6.5e-3."""
    kind, dtype = case["kind"], case.get("dtype")
    if kind == "quantised":
        return "exact"  # integer sums, one defined rounding
    if kind == "tower":
        return {"rel": {"f32": 8e-6, "f16": 3e-3, "bf16": 2.5e-2}[dtype]}
    if kind == "stages":
        return {"rel": {"f32": 1e-5, "f16": 2e-3, "bf16": 7e-3}[dtype]}
    if kind == "weight_gradient":
        return {"rel": {"f32": 3.5e-5, "f16": 2e-3, "bf16": 7e-3}[dtype]}
    return {"rel": {"f32": 4e-6, "f16": 1.4e-3, "bf16": 7e-3}[dtype]}

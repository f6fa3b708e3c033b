"""What a program asks of this library, as timed cases.

A case is one pass through the public entry points.  The matrix products, batched products and element-wise chains go
through the C ABI with tensors resident and descriptors marshalled once, as a compiled host program calls it; the layers
(Dense with its pullback, the LSTM cell) go through the operators of the package, which allocate their results.  Sizes are
those of the benchmark and the tests, or generic ones in between; `draw` spreads them over the ranges the listed cases
stand for, odd extents among them.
"""
import ctypes
import math

import torch

import swiftrt_amd as srt
from swiftrt_amd import native

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
STORAGE = {"f32": "float32", "f16": "float16", "bf16": "uint16"}
TYPESTR = {"float32": "<f4", "float16": "<f2", "uint16": "<i2"}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
# extents a drawn problem may have: its matrix time stays below the largest listed product's
MOST_FLOPS = {"f32": 1.0e11, "f16": 1.0e12, "bf16": 1.0e12}
MOST_ELEMENTS = 4096 * 11008


def product(name, dtype, m, n, k, batch=1, ta=False, tb=False, bias=False, act="identity"):
    return {"name": name, "kind": "product", "dtype": dtype, "batch": batch, "m": m, "n": n, "k": k, "ta": ta, "tb": tb,
            "bias": bias, "act": act}


def listed():
    return [
        # a small product in the default element type: latency of one launch
        product("f32_512", "f32", 512, 512, 512),
        # a batch of small half-precision products against transposed right operands
        product("batch_f16_32x256", "f16", 256, 256, 256, batch=32, tb=True),
        # scores of 64 query / key blocks: a short k loop, bound by writing the result
        product("batch_bf16_64x512x64", "bf16", 512, 512, 64, batch=64, tb=True),
        # the large product
        product("bf16_8192", "bf16", 8192, 8192, 8192),
        # prompt-sized product: a quarter of a device's worth of 256 x 256 tiles
        product("bf16_1024x4096", "bf16", 1024, 4096, 4096),
        # a projection onto an odd number of classes: no row of the weight or of the result keeps an alignment
        product("bf16_2048x50257x768", "bf16", 2048, 50257, 768),
        # one decoding step for eight sequences against a pre-transposed weight: bound by reading the weight
        product("decode_bf16_m8", "bf16", 8, 14336, 4096, tb=True),
        # serving 32 requests through a Dense layer in the layer's own weight layout
        product("dense_bf16_m32", "bf16", 32, 11008, 4096, bias=True, act="relu"),
        # a training step of a Dense layer: forward, then both gradients and the bias gradient
        {"name": "train_bf16_4096x11008", "kind": "train", "dtype": "bf16", "batch": 4096, "inputs": 4096, "outputs": 11008,
         "act": "relu"},
        # the same for a small layer in the default element type
        {"name": "train_f32_256x784", "kind": "train", "dtype": "f32", "batch": 256, "inputs": 784, "outputs": 1000,
         "act": "tanh"},
        # one step of an LSTM cell
        {"name": "lstm_f32_64x512", "kind": "lstm", "dtype": "f32", "batch": 64, "inputs": 512, "hidden": 512},
        # the unfused tail of a Dense layer: bias broadcast over the rows, then the activation
        {"name": "map_bf16_bias_tanh", "kind": "map", "op": "bias_tanh", "dtype": "bf16", "m": 4096, "n": 11008},
    ]


# ---- drawn cases ---------------------------------------------------------------------------------------------------
def _extent(rng, low, high):
    """Log-uniform in [low, high]; most extents are whole units of 64 or 8, the others are whatever comes."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    unit = rng.choice((64, 64, 8, 1))
    return min(high, max(low, v // unit * unit))


def _product(rng, dtype):
    batch = 1
    while True:
        if rng.random() < 0.25:
            batch = _extent(rng, 2, 64)
            m, n, k = _extent(rng, 32, 1024), _extent(rng, 32, 1024), _extent(rng, 32, 2048)
        elif rng.random() < 0.33:
            m, n, k = rng.choice((1, 2, 4, 8, 16, 32, _extent(rng, 1, 64))), _extent(rng, 512, 14336), _extent(rng, 256, 8192)
        else:
            m, n, k = _extent(rng, 64, 8192), _extent(rng, 64, 16384), _extent(rng, 64, 8192)
        if 2.0 * batch * m * n * k <= MOST_FLOPS[dtype] and batch * max(m * n, m * k, n * k) <= 3 * MOST_ELEMENTS:
            break
    act = rng.choice(("identity", "identity", "identity", "relu", "tanh", "sigmoid"))
    return {"kind": "product", "dtype": dtype, "batch": batch, "m": m, "n": n, "k": k, "ta": m > 64 and rng.random() < 0.3,
            "tb": rng.random() < 0.5, "bias": act != "identity" or rng.random() < 0.2, "act": act}


def draw(rng):
    kind = rng.choice(("product", "product", "product", "product", "train", "lstm", "map", "map"))
    dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
    if kind == "product":
        return _product(rng, dtype)
    if kind == "train":
        while True:
            b, i, o = _extent(rng, 8, 4096), _extent(rng, 64, 8192), _extent(rng, 64, 11008)
            if 6.0 * b * i * o <= MOST_FLOPS[dtype] and max(b * o, i * o) <= MOST_ELEMENTS:
                break
        return {"kind": kind, "dtype": dtype, "batch": b, "inputs": i, "outputs": o,
                "act": rng.choice(("relu", "relu", "tanh", "sigmoid"))}
    if kind == "lstm":
        return {"kind": kind, "dtype": dtype, "batch": _extent(rng, 1, 512), "inputs": _extent(rng, 32, 1024),
                "hidden": _extent(rng, 32, 1024)}
    while True:
        m, n = _extent(rng, 256, 16384), _extent(rng, 256, 16384)
        if MOST_ELEMENTS // 16 <= m * n <= MOST_ELEMENTS:
            break
    return {"kind": kind, "op": rng.choice(("bias_tanh", "residual", "cast", "transpose")), "dtype": dtype, "m": m, "n": n}


# ---- tensors -------------------------------------------------------------------------------------------------------
class _Device:
    """A resident tensor's memory as torch sees it; holds the tensor."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tensor.shape, "strides": None, "version": 2, "typestr": TYPESTR[str(tensor.dtype)],
            "data": (tensor.device_read(srt.current_queue()), False)}


def _torch(tensor, dtype):
    """The dense result `tensor` as a torch tensor over the same device memory."""
    t = torch.as_tensor(_Device(tensor), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bf16" else t


class _Inputs:
    """Seeded values made on the device, moved into resident tensors of the library."""

    def __init__(self, dtype, seed):
        self.dtype, self.queue = dtype, srt.current_queue()
        self.rng = torch.Generator(device="cuda")
        self.rng.manual_seed(int(seed))

    def _resident(self, values):
        values = values.to(TORCH[self.dtype]).contiguous()
        t = self.empty(values.shape)
        ptr = t.device_read_write(self.queue)
        torch.cuda.synchronize()
        native.check(native.lib().srtMemcpyAsync(ctypes.c_void_p(ptr), ctypes.c_void_p(values.data_ptr()),
                                                 values.numel() * values.element_size(), native.D2D, self.queue.stream))
        self.queue.wait_for_completion()
        return t

    def normal(self, shape, scale=1.0):
        return self._resident(torch.randn(shape, generator=self.rng, device="cuda") * scale)

    def uniform(self, shape, bound):
        return self._resident((torch.rand(shape, generator=self.rng, device="cuda") * 2 - 1) * bound)

    def empty(self, shape, dtype=None):
        return srt.Tensor(shape=list(shape), dtype=STORAGE[dtype or self.dtype])


def _call(name, *args):
    """One native call with its arguments marshalled: tensors become a pointer and a descriptor."""
    queue, argv, keep = srt.current_queue(), [], []
    for a in args:
        if isinstance(a, srt.Tensor):
            descriptor, storage = a.descriptor()
            argv += [a.device_read(queue), ctypes.byref(descriptor)]
            keep.append((a, descriptor, storage))
        elif a is None:
            argv += [None, None]
        else:
            argv.append(a)
    fn = getattr(native.lib(), name)

    def call():
        native.check(fn(*argv, queue.stream), name)
    call.keep = keep
    return call


# ---- the paths -----------------------------------------------------------------------------------------------------
def _prepare_product(c, make):
    lead = [c["batch"]] if c["batch"] > 1 else []
    m, n, k = c["m"], c["n"], c["k"]
    a = make.normal(lead + ([k, m] if c["ta"] else [m, k]))
    b = make.normal(lead + ([n, k] if c["tb"] else [k, n]), 1 / math.sqrt(k))
    bias = make.uniform([n], 0.1) if c["bias"] else None
    out = make.empty(lead + [m, n])
    out.device_read_write(make.queue)
    call = _call("srtMatmulBiasActivation", a, int(c["ta"]), b, int(c["tb"]), bias, int(srt.ActivationType[c["act"]]), 0.0, out)
    return {"calls": [call], "out": [_torch(out, c["dtype"])]}


def _prepare_map(c, make):
    m, n, dtype = c["m"], c["n"], c["dtype"]
    x = make.normal([m, n])
    if c["op"] == "bias_tanh":
        bias, z, y = make.uniform([n], 0.1), make.empty([m, n]), make.empty([m, n])
        outs = [(z, dtype), (y, dtype)]
        calls = [_call("srtAdd", x, srt.Tensor.repeating(bias, [m, n]), z), _call("srtTanh", z, y)]
    elif c["op"] == "residual":
        other, y = make.normal([m, n]), make.empty([m, n])
        outs = [(y, dtype)]
        calls = [_call("srtAdd", x, other, y)]
    elif c["op"] == "cast":
        to = "bf16" if dtype == "f32" else "f32"
        y = make.empty([m, n], to)
        outs = [(y, to)]
        calls = [_call("srtCopy", x, y)]
    else:   # a transposed view made dense
        y = make.empty([n, m])
        outs = [(y, dtype)]
        calls = [_call("srtCopy", x.t, y)]
    return {"calls": calls, "out": [_torch(t, d) for t, d in outs]}


def _prepare_train(c, make):
    b, i, o = c["batch"], c["inputs"], c["outputs"]
    layer = srt.Dense(make.normal([i, o], 1 / math.sqrt(i)), make.uniform([o], 0.1), srt.ActivationType[c["act"]])
    return {"layer": layer, "x": make.normal([b, i]), "dy": make.normal([b, o], 1 / math.sqrt(o)), "dtype": c["dtype"]}


def _run_train(s):
    y = s["layer"](s["x"])
    dx, dw, db = srt.dense_backward(s["layer"], s["x"], y, s["dy"])
    return {k: _torch(t, s["dtype"]) for k, t in (("y", y), ("dx", dx), ("dw", dw), ("db", db))}


def _prepare_lstm(c, make):
    b, i, h = c["batch"], c["inputs"], c["hidden"]
    cell = srt.LSTMCell(make.normal([i + h, 4 * h], 1 / math.sqrt(i + h)), make.uniform([4 * h], 0.1))
    return {"cell": cell, "x": make.normal([b, i]), "c": make.normal([b, h], 0.5), "h": make.uniform([b, h], 0.9),
            "dtype": c["dtype"]}


def _run_lstm(s):
    new_cell, new_hidden = s["cell"](s["x"], s["c"], s["h"])
    return {"cell": _torch(new_cell, s["dtype"]), "hidden": _torch(new_hidden, s["dtype"])}


def _run_calls(s):
    for call in s["calls"]:
        call()
    return s["out"]


PREPARE = {"product": _prepare_product, "map": _prepare_map, "train": _prepare_train, "lstm": _prepare_lstm}
RUN = {"product": _run_calls, "map": _run_calls, "train": _run_train, "lstm": _run_lstm}


def prepare(case, seed):
    state = PREPARE[case["kind"]](case, _Inputs(case["dtype"], seed))
    state["kind"] = case["kind"]
    return state


def run(state):
    return RUN[state["kind"]](state)


def work(case):
    e = SIZE[case["dtype"]]
    if case["kind"] == "product":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return {"bytes": e * (b * (m * k + k * n + m * n) + (n if case["bias"] else 0)), "flops": 2.0 * b * m * n * k}
    if case["kind"] == "train":
        b, i, o = case["batch"], case["inputs"], case["outputs"]
        # in: x, W, bias, dy; out: y, dx, dW, dbias
        return {"bytes": e * (2 * b * i + 2 * i * o + 2 * o + 2 * b * o), "flops": 6.0 * b * i * o}
    if case["kind"] == "lstm":
        b, i, h = case["batch"], case["inputs"], case["hidden"]
        # in: x, cell, hidden, weight, bias; out: cell, hidden
        return {"bytes": e * (b * (i + 4 * h) + (i + h) * 4 * h + 4 * h), "flops": 8.0 * b * (i + h) * h}
    m, n = case["m"], case["n"]
    if case["op"] == "bias_tanh":   # both tensors are results
        return {"bytes": e * (3 * m * n + n), "flops": 2.0 * m * n}
    if case["op"] == "residual":
        return {"bytes": e * 3 * m * n, "flops": 1.0 * m * n}
    if case["op"] == "cast":
        return {"bytes": m * n * (e + (2 if case["dtype"] == "f32" else 4)), "flops": 0}
    return {"bytes": e * 2 * m * n, "flops": 0}


# about four times the largest relative errors seen against the same path in 64 bits (2-norm; largest element), results and
# what the path itself stores in between rounded to the element type
TOLERANCE = {
    "product": {"f32": (3.5e-6, 4e-5), "f16": (8.5e-4, 2e-3), "bf16": (6.7e-3, 1.6e-2)},
    "lstm": {"f32": (3.5e-6, 4e-5), "f16": (2e-3, 1.2e-2), "bf16": (1.6e-2, 1e-1)},   # eight roundings after the gates
    "train": {"f32": (3.5e-6, 4e-5), "f16": (1.5e-3, 7e-3), "bf16": (1e-2, 3.6e-2)},
    # a pre-activation within rounding of zero may fall on either side, and a whole gradient entry with it
    "train relu": {"f32": (3e-3, 6e-1), "f16": (3e-3, 6e-1), "bf16": (7e-3, 6e-1)},
}


def tolerance(case):
    kind = case["kind"]
    if kind == "map":
        if case["op"] != "bias_tanh":
            return "exact"
        kind = "product"
    elif kind == "train" and case["act"] == "relu":
        kind = "train relu"
    rel, most = TOLERANCE[kind][case["dtype"]]
    return {"rel": rel, "max": most}

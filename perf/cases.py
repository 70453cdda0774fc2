"""The work that programs built on this package have it do, as cases that can be timed.

Two ways lead into the package: a `dl::Model` made from a graph (the five workloads of `esp-dl_amd/zoo.py`, single
layers and the attention block of exported detectors), run as a HIP graph on batches that lie in HBM or arrive from
host memory, and the kernel C ABI called operator by operator on tensors.  Inputs are seeded uniform int8 / int16, as
`bench.py` and the tests use them; a network's weights are those its zoo function draws (a deployed model is a fixed
file, what changes from pass to pass is the batch).
"""
import functools
import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("esp-dl_amd")
zoo = pkg.zoo

_LISTED = [
    # one 3x3 layer at one image: the smallest call there is, a single launch (the first benchmark configuration)
    {"name": "conv_56x56_c64_b1", "kind": "conv", "h": 56, "w": 56, "cin": 64, "cout": 64, "k": 3, "stride": 1, "s16": False, "batch": 1},
    # the same layer over a batch: ordinary dense convolution work
    {"name": "conv_56x56_c64_b256", "kind": "conv", "h": 56, "w": 56, "cin": 64, "cout": 64, "k": 3, "stride": 1, "s16": False, "batch": 256},
    # a layer whose sizes are multiples of nothing (the odd row of the operator test matrix): pruned or hand-made networks
    {"name": "conv_19x23_c22_oc33_b200", "kind": "conv", "h": 19, "w": 23, "cin": 22, "cout": 33, "k": 3, "stride": 1, "s16": False, "batch": 200},
    # one inverted-residual block with its Clips: a mobile network's unit (the second configuration)
    {"name": "block_b256", "kind": "block", "batch": 256},
    # a classifier asked for one picture at a time, picture and scores in host memory: latency as a camera loop sees it
    {"name": "mobilenetv2_224_b1_host", "kind": "mobilenetv2", "resolution": 224, "batch": 1, "half_even": False, "host": True},
    # the classifier over a full batch that lies in HBM: the headline workload (the third configuration)
    {"name": "mobilenetv2_224_b256", "kind": "mobilenetv2", "resolution": 224, "batch": 256, "half_even": False, "host": False},
    # a smaller resolution, an odd batch, and the rounding of files exported for the ESP32-P4
    {"name": "mobilenetv2_160_b37_even", "kind": "mobilenetv2", "resolution": 160, "batch": 37, "half_even": True, "host": False},
    # the detector over a batch of full-size frames, int16 head included: the most work (the fourth configuration)
    {"name": "yolo_640_b64", "kind": "yolo", "resolution": 640, "batch": 64},
    # the detector on one frame: some sixty dependent launches
    {"name": "yolo_416_b1", "kind": "yolo", "resolution": 416, "batch": 1},
    # the text-line recognizer over a page's worth of crops (the fifth configuration)
    {"name": "ocr_b512", "kind": "ocr", "batch": 512},
    # the attention block of exported detectors on a 20 x 20 map: activation products, softmax, transposes
    {"name": "attention_20_b32", "kind": "attention", "hw": 20, "heads": 2, "batch": 32},
    # operators called one by one through the C ABI on tensors, as a program with its own graph does
    {"name": "ops_56x56_c144_b256", "kind": "ops", "h": 56, "w": 56, "c": 144, "batch": 256},
]


def listed():
    return [dict(c) for c in _LISTED]


def _log(rng, lo, hi):
    """A whole number of lo .. hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["conv", "conv", "conv", "block", "mobilenetv2", "mobilenetv2", "yolo", "yolo", "ocr", "attention", "ops", "ops"])
    if kind == "conv":
        s16 = rng.random() < 0.2
        c = {"kind": kind, "h": _log(rng, 7, 112), "w": _log(rng, 7, 112), "cin": _log(rng, 3, 256), "cout": _log(rng, 8, 256),
             "k": rng.choice([1, 1, 3, 3, 3, 5]), "stride": rng.choice([1, 1, 2]), "s16": s16, "batch": 1}
        if rng.random() < 0.6:  # most networks keep their channels at multiples of 16; the others do not
            c["cin"], c["cout"] = max(16, c["cin"] // 16 * 16), max(16, c["cout"] // 16 * 16)
        w = work(c)
        top = min(256, 4e8 / w["bytes"], (1e10 if s16 else 2e11) / w["flops"])
        c["batch"] = _log(rng, 1, max(1, int(top)))
        return c
    if kind == "block":
        return {"kind": kind, "batch": _log(rng, 1, 300)}
    if kind == "mobilenetv2":
        res = 32 * rng.randint(3, 7)
        host = rng.random() < 0.3
        return {"kind": kind, "resolution": res, "batch": _log(rng, 1, 8 if host else 256), "half_even": rng.random() < 0.35, "host": host}
    if kind == "yolo":
        res = 32 * rng.randint(10, 20)
        return {"kind": kind, "resolution": res, "batch": _log(rng, 1, 64)}
    if kind == "ocr":
        return {"kind": kind, "batch": _log(rng, 1, 512)}
    if kind == "attention":
        return {"kind": kind, "hw": rng.randint(7, 22), "heads": rng.randint(1, 4), "batch": _log(rng, 1, 32)}
    c = {"kind": kind, "h": _log(rng, 7, 80), "w": _log(rng, 7, 80), "c": _log(rng, 16, 256)}
    if rng.random() < 0.6:
        c["c"] = c["c"] // 16 * 16
    c["batch"] = _log(rng, 1, min(256, int(1.15e8 / (c["h"] * c["w"] * c["c"]))))
    return c


@functools.lru_cache(maxsize=None)
def _spec_of(items):
    """The graph of a case: what a program reads from its model file."""
    c = dict(items)
    kind = c["kind"]
    if kind == "block":
        return zoo.config2_mbv2_block()
    if kind == "mobilenetv2":
        return zoo.config3_mobilenetv2(resolution=c["resolution"])
    if kind == "yolo":
        return zoo.config4_yolo_style(resolution=c["resolution"])
    if kind == "ocr":
        return zoo.config5_ocr_style()
    if kind == "attention":
        return zoo.attention_block(hw=c["hw"], heads=c["heads"], key_dim=32, head_dim=64)
    g = zoo.GraphSpec("single_conv")
    b = zoo.Builder(g, 0xE5D1, per_channel=True, w_exp_range=None)
    s16 = c["s16"]
    x = b.input("input", [1, c["h"], c["w"], c["cin"]], -12 if s16 else -5, zoo.INT16 if s16 else zoo.INT8)
    b.output(b.conv(x, c["cout"], k=c["k"], stride=c["stride"], relu=True, s16=s16, name="conv"))
    return g


def _spec(case):
    return _spec_of(tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "batch", "half_even", "host"))))


class _DeviceArray:
    """A tensor of a model where it lies in HBM, for torch.as_tensor (which keeps this object, and so the model)."""

    def __init__(self, mdl, name):
        self.owner = mdl
        typestr = "<i2" if mdl.graph_spec.dtype(name) == zoo.INT16 else "|i1"
        ptr = pkg.model.lib().espdl_model_tensor_device_ptr(mdl.h, name.encode())
        self.__cuda_array_interface__ = {"version": 3, "shape": tuple(mdl.shape(name)), "typestr": typestr, "data": (ptr, False), "strides": None}


def _view(mdl, name):
    return torch.as_tensor(_DeviceArray(mdl, name), device="cuda")


@functools.lru_cache(maxsize=None)
def _stream():
    """The one stream on which a serving program runs its models."""
    return torch.cuda.Stream()


def _randint(gen, shape, dtype):
    lim = 32768 if dtype == torch.int16 else 128
    return torch.randint(-lim, lim, shape, dtype=dtype, device="cuda", generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if case["kind"] == "ops":
        return _prepare_ops(case, gen)
    spec = _spec(case)
    mdl = pkg.model.Model(pkg.model.Graph.from_spec(spec), case["batch"], round_mode=1 if case.get("half_even") else 0,
                          stream=_stream().cuda_stream)
    mdl.graph_spec = spec
    if not mdl.enable_graph():
        raise RuntimeError("the plan could not be captured")
    name = spec.inputs[0]
    if case.get("host"):
        shape = [case["batch"]] + spec.shape(name)[1:]
        x = np.random.default_rng(seed).integers(-128, 128, size=shape, dtype=np.int8)
        return {"model": mdl, "host_input": x, "input": name, "output": spec.outputs[0]}
    x = _view(mdl, name)
    x.copy_(_randint(gen, tuple(x.shape), x.dtype))
    torch.cuda.synchronize()
    return {"model": mdl, "outputs": {n: _view(mdl, n) for n in spec.outputs}}


def _prepare_ops(case, gen):
    n, h, w, c = case["batch"], case["h"], case["w"], case["c"]
    x = _randint(gen, (n, h, w, c), torch.int8)
    weights = np.random.default_rng(0xE5D2)
    dev = lambda a, t: torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=t)  # noqa: E731
    s = {
        "x": x,
        "filter": dev(weights.integers(-128, 128, size=(3, 3, c)), torch.int8),
        "bias": dev(weights.integers(-4096, 4097, size=c), torch.int32),
        "shift": dev(weights.integers(6, 11, size=c), torch.int32),
        "slope": dev(weights.integers(-128, 128, size=c), torch.int8),
        "table": dev(zoo.make_lut(zoo.silu, -5, -5), torch.int8),
    }
    for name in ("conv", "prelu", "add", "pool"):
        s[name] = torch.empty_like(x)
    for name in ("concat", "lut"):
        s[name] = torch.empty((n, h, w, 2 * c), dtype=torch.int8, device="cuda")
    return s


def run(state):
    if "model" not in state:
        return _run_ops(state)
    mdl = state["model"]
    if "host_input" in state:
        mdl.set_input(state["input"], state["host_input"])
        mdl.run()
        return mdl.get_tensor(state["output"])
    mdl.run_async()
    return state["outputs"]


def _run_ops(s):
    """Depthwise 3x3 -> PReLU -> residual Add -> 5x5 max pool -> Concat with its input -> table activation."""
    y = pkg.conv2d(s["x"], s["filter"], s["bias"], s["shift"], (3, 3), pads=(1, 1, 1, 1), depthwise=True, out=s["conv"])
    p = pkg.prelu_s8(y, s["slope"], 7, out=s["prelu"])
    a = pkg.add_s8(p, s["x"], out=s["add"])
    m = pkg.max_pool(a, (5, 5), (1, 1), (2, 2, 2, 2), out=s["pool"])
    c = pkg.concat([a, m], 3, out=s["concat"])
    t = pkg.lut_s8(c, s["table"], out=s["lut"])
    return [y, p, a, m, c, t]


def work(case):
    n = case["batch"]
    if case["kind"] == "ops":
        size = n * case["h"] * case["w"] * case["c"]
        # every call reads its operands and writes its result: 2 + 2 + 3 + 2 + 4 + 4 tensors of the input's size
        return {"bytes": 17 * size + 18 * case["c"], "flops": 18 * size}
    spec = _spec(case)
    width = {zoo.FLOAT: 4, zoo.INT8: 1, zoo.INT16: 2, zoo.INT32: 4, zoo.INT64: 8}
    values = sum(int(np.prod(spec.shape(t))) * width[spec.dtype(t)] for t in spec.inputs + spec.outputs)
    constants = sum(data.nbytes for _, _, data, _ in spec.initializers.values())
    return {"bytes": n * values + constants, "flops": 2 * n * spec.macs_per_image}


def tolerance(case):
    """Integer arithmetic with defined rounding: every byte is fixed.  (The float32 softmax inside the attention block
    sums in a defined order and its result leaves the block as int8.)"""
    return "exact"

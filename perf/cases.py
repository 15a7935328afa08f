"""Workloads of this backend as a user's program runs them, for timing one pass of each.

Four kinds, all through the package's public entry points:

  network  ResNet-18 compiled from its Relay graph by the host layer (fp32, or quantised to int8), the way bench.py
           runs it: weights frozen or re-read in every run, launches enqueued one by one or replayed as a graph
  conv     nn_conv2d on its own, fp32, with its fused epilogue (bias, residual, ReLU)
  qconv    the quantised convolution on its own, int8 on the channel-blocked layout, weights packed beforehand
  dense    nn_gemm / nn_dense with bias
  stream   the bandwidth-bound operators in a row: 3x3/2 max pool, residual add + ReLU, global average pool

A compiled module, packed weights and the stream a serving loop uses are made by prepare(), as a program makes them
once; everything that a new input needs is in run().
"""
import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("hdkx-aicompiler_amd")
hostapi = importlib.import_module("hdkx-aicompiler_amd.hostapi")
resnet18 = importlib.import_module("hdkx-aicompiler_amd.resnet18")
qresnet18 = importlib.import_module("hdkx-aicompiler_amd.qresnet18")
synth = importlib.import_module("hdkx-aicompiler_amd.synth")


def listed():
    return [
        # One image at a time behind an interactive service: latency of a chain of small launches, replayed as a graph.
        {"name": "net_f32_b1", "kind": "network", "dtype": "f32", "batch": 1, "hw": 224, "frozen": True, "graph": True},
        # Throughput serving: the batch the framework is benchmarked on.
        {"name": "net_f32_b64", "kind": "network", "dtype": "f32", "batch": 64, "hw": 224, "frozen": True, "graph": False},
        # What a caller gets who only switched the target: weights re-read in every run; a partly filled batch of
        # images whose size is not the usual one, so that every layer's map is odd.
        {"name": "net_f32_b6_odd", "kind": "network", "dtype": "f32", "batch": 6, "hw": 193, "frozen": False, "graph": False},
        # The quantised network at the benchmarked batch.
        {"name": "net_i8_b64", "kind": "network", "dtype": "i8", "batch": 64, "hw": 224, "frozen": True, "graph": False},
        # The quantised network on a handful of smaller images, replayed as a graph.
        {"name": "net_i8_b5", "kind": "network", "dtype": "i8", "batch": 5, "hw": 160, "frozen": True, "graph": True},
        # One convolution called by itself (benchmark configuration 1): the smallest call, mostly its launch.
        {"name": "conv_3x3_b1", "kind": "conv", "n": 1, "c": 64, "h": 56, "w": 56, "o": 64, "k": 3, "stride": 1, "residual": False, "relu": True},
        # The same operator where nothing is a round number.
        {"name": "conv_3x3_ragged", "kind": "conv", "n": 7, "c": 90, "h": 37, "w": 51, "o": 150, "k": 3, "stride": 1, "residual": True, "relu": True},
        # A pointwise convolution that widens a mid-sized map.
        {"name": "conv_1x1", "kind": "conv", "n": 32, "c": 128, "h": 28, "w": 28, "o": 512, "k": 1, "stride": 1, "residual": True, "relu": True},
        # A filter size the ResNet graph does not hold.
        {"name": "conv_5x5", "kind": "conv", "n": 8, "c": 64, "h": 27, "w": 27, "o": 96, "k": 5, "stride": 1, "residual": False, "relu": True},
        # One quantised layer in the middle of a network, with its residual.
        {"name": "qconv_3x3", "kind": "qconv", "n": 32, "c": 128, "h": 28, "w": 28, "o": 128, "k": 3, "stride": 1, "residual": True, "relu": True},
        # A wide dense layer on a ragged batch.
        {"name": "dense", "kind": "dense", "m": 300, "n": 1000, "k": 2048, "trans_b": True},
        # The bandwidth-bound operators at the first layer's shape (benchmark configuration 2).
        {"name": "stream_112", "kind": "stream", "n": 64, "c": 64, "h": 112, "w": 112},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["network", "conv", "qconv", "dense", "stream"], [8, 6, 2, 2, 2])[0]
    if kind == "network":
        # from a thumbnail to the usual 224 pixels, one image to a full batch
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "i8"]), "batch": _log_int(rng, 1, 64), "hw": rng.randint(64, 224),
                "frozen": rng.random() < 0.7, "graph": rng.random() < 0.4}
    if kind == "conv":
        while True:
            k = rng.choice([1, 3, 3, 3, 5, 7])
            case = {"kind": kind, "n": _log_int(rng, 1, 64), "c": _log_int(rng, 3, 512), "h": _log_int(rng, 7, 112), "w": _log_int(rng, 7, 112),
                    "o": _log_int(rng, 16, 512), "k": k, "stride": rng.choice([1, 1, 2]), "residual": rng.random() < 0.5, "relu": rng.random() < 0.7}
            if rng.random() < 0.5:      # half of all layers have the channel counts networks are usually built with
                case["c"], case["o"] = max(16, case["c"] // 16 * 16), max(16, case["o"] // 16 * 16)
            if 1e7 <= work(case)["flops"] <= 4e9:
                return case
    if kind == "qconv":
        while True:
            case = {"kind": kind, "n": _log_int(rng, 1, 64), "c": 16 * _log_int(rng, 1, 32), "h": _log_int(rng, 7, 56), "w": _log_int(rng, 7, 56),
                    "o": 32 * _log_int(rng, 1, 16), "k": rng.choice([1, 3, 3]), "stride": rng.choice([1, 1, 2]), "residual": rng.random() < 0.5,
                    "relu": rng.random() < 0.7}
            if 1e7 <= work(case)["flops"] <= 15e9:
                return case
    if kind == "dense":
        k = _log_int(rng, 32, 4096)
        return {"kind": kind, "m": _log_int(rng, 1, 512), "n": _log_int(rng, 10, 4096), "k": k if rng.random() < 0.3 else max(32, k // 32 * 32),
                "trans_b": rng.random() < 0.8}
    return {"kind": kind, "n": _log_int(rng, 1, 64), "c": _log_int(rng, 16, 64), "h": rng.randint(14, 112), "w": rng.randint(14, 112)}


# ---- inputs

def _random(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    normal = lambda shape, sigma=1.0: torch.randn(shape, generator=g, device="cuda") * sigma
    uniform = lambda shape, lo, hi: torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo
    int8 = lambda shape: torch.randint(-127, 128, shape, generator=g, device="cuda", dtype=torch.int8)
    return normal, uniform, int8


def _weights(normal, shape):
    return normal(shape, math.sqrt(2.0 / math.prod(shape[1:])))


def _network_constants(normal, uniform):
    return [_weights(normal, s) if len(s) > 1 else uniform(s, -0.1, 0.1) for s in synth.resnet18_const_shapes()]


def _activation_ranges():
    """max |activation| of every quantised tensor, from the second moments of a network with Kaiming weights on N(0, 1)
    input (a ReLU halves the second moment that its convolution doubles; a block adds its identity), at 5 sigma."""
    peak = lambda moment: 5.0 * math.sqrt(2.0 * moment)
    amax = {"input": 5.0, "conv1": peak(1.0)}
    moment = 2.0        # behind the max pool
    for stage in range(4):
        for block in range(2):
            name = "l%d.%d" % (stage + 1, block)
            first = block == 0 and stage > 0
            amax[name + ".conv1"] = peak(moment)
            if first:
                amax[name + ".down"] = peak(moment)
            moment = moment + (moment if first else 0.5 * moment)
            amax[name + ".conv2"] = peak(moment)
    amax["gap"] = math.sqrt(2.0 * moment)
    return amax


class _Network:
    """A compiled network with the buffers that a serving program binds to it."""

    _stream = None

    def __init__(self, module, tensors, out, case):
        self.module, self.tensors, self.out = module, tensors, out
        if case["frozen"]:
            module.freeze_constants(True)
        self.stream = torch.cuda.current_stream().cuda_stream
        if case["graph"]:
            # replay needs a stream of the caller's: one for the whole program, as a serving loop has
            if _Network._stream is None:
                _Network._stream = torch.cuda.Stream()
            self.stream = _Network._stream.cuda_stream
            module.enable_graph_replay(True)
        self.args = module.packed(tensors)

    def __del__(self):
        try:
            self.module.close()
        except Exception:
            pass


def prepare(case, seed):
    normal, uniform, int8 = _random(seed)
    kind = case["kind"]
    if kind == "network":
        batch, hw = case["batch"], case["hw"]
        consts = _network_constants(normal, uniform)
        x = normal((batch, 3, hw, hw))
        out = torch.empty((batch, 1000), device="cuda")
        if case["dtype"] == "f32":
            module = hostapi.CompiledResNet18(batch, hw, "hip", sync_after_run=False)
        else:
            model = qresnet18.prepare([c.cpu().numpy() for c in consts], _activation_ranges())
            module = hostapi.CompiledQResNet18(model, batch, hw, "hip", sync_after_run=False)
            consts = [torch.from_numpy(np.ascontiguousarray(c)).cuda() for c in module.constants(model)]
        return _Network(module, [x] + consts + [out], out, case)
    if kind == "conv":
        n, c, h, w, o, k = (case[f] for f in ("n", "c", "h", "w", "o", "k"))
        oh, ow = _out(h, k, case["stride"]), _out(w, k, case["stride"])
        return {"x": normal((n, c, h, w)).relu_(), "w": _weights(normal, (o, c, k, k)), "bias": uniform((o,), -0.1, 0.1),
                "residual": normal((n, o, oh, ow)).relu_() if case["residual"] else None,
                "stride": case["stride"], "pad": k // 2, "relu": case["relu"]}
    if kind == "qconv":
        n, c, h, w, o, k = (case[f] for f in ("n", "c", "h", "w", "o", "k"))
        oh, ow = _out(h, k, case["stride"]), _out(w, k, case["stride"])
        weights = int8((o, c, k, k))
        return {"x": pkg.i8_nchw_to_c16(int8((n, c, h, w)).clamp_(min=0)), "c": c, "w": pkg.qconv2d_c16_pack_weights(weights), "w_shape": (o, c, k, k),
                "bias": torch.randint(-2000, 2000, (o,), device="cuda", dtype=torch.int32, generator=torch.Generator(device="cuda").manual_seed(seed + 1)),
                "mult": uniform((o,), 0.5, 1.5) / (73.0 * 52.0 * math.sqrt(c * k * k / 2.0) / 40.0),
                "residual": pkg.i8_nchw_to_c16(int8((n, o, oh, ow)).clamp_(min=0)) if case["residual"] else None,
                "stride": case["stride"], "pad": k // 2, "relu": case["relu"]}
    if kind == "dense":
        m, n, k = case["m"], case["n"], case["k"]
        b = _weights(normal, (n, k))
        return {"a": normal((m, k)).relu_(), "b": b if case["trans_b"] else b.t().contiguous(), "bias": uniform((n,), -0.1, 0.1),
                "trans_b": 1 if case["trans_b"] else 0}
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    return {"x": uniform((n, c, h, w), -1.0, 1.0), "skip": uniform((n, c, (h + 1) // 2, (w + 1) // 2), -1.0, 1.0)}


def run(state):
    if isinstance(state, _Network):
        state.module.run_packed(state.args, state.stream)
        return state.out
    s = state
    if "mult" in s:
        return pkg.qconv2d_c16(s["x"], s["c"], s["w"], s["w_shape"], s["bias"], s["mult"], s["residual"], 0.25, s["stride"], s["pad"], s["relu"])
    if "w" in s:
        return pkg.conv2d(s["x"], s["w"], s["bias"], s["residual"], s["stride"], s["pad"], 1, s["relu"])
    if "trans_b" in s:
        return pkg.gemm(s["a"], s["b"], s["bias"], 1.0, 1.0, s["trans_b"])
    pooled = pkg.pool2d(s["x"], 3, 2, 1)
    y = pkg.binary(0, pooled, s["skip"], True)
    return pooled, y, pkg.global_avg_pool2d(y)


# ---- what a pass cannot do without

def _out(size, k, stride):
    return (size + 2 * (k // 2) - k) // stride + 1


def work(case):
    kind = case["kind"]
    if kind == "network":
        batch, hw = case["batch"], case["hw"]
        params = sum(math.prod(s) for s in synth.resnet18_const_shapes())
        return {"bytes": 4 * batch * (3 * hw * hw + 1000) + params * (4 if case["dtype"] == "f32" else 1), "flops": batch * resnet18.flops_per_image(hw)}
    if kind in ("conv", "qconv"):
        n, c, h, w, o, k = (case[f] for f in ("n", "c", "h", "w", "o", "k"))
        outputs = n * o * _out(h, k, case["stride"]) * _out(w, k, case["stride"])
        size = 4 if kind == "conv" else 1
        return {"bytes": size * (n * c * h * w + o * c * k * k + outputs * (2 if case["residual"] else 1)) + 8 * o, "flops": 2 * outputs * c * k * k}
    if kind == "dense":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + n * k + n + m * n), "flops": 2 * m * n * k}
    planes, h, w = case["n"] * case["c"], case["h"], case["w"]
    pooled = planes * ((h + 1) // 2) * ((w + 1) // 2)
    # (the pooled map and the sum are results; both are written once)
    return {"bytes": 4 * (planes * h * w + 3 * pooled + planes), "flops": 9 * pooled + 3 * pooled}


def tolerance(case):
    if case["kind"] == "qconv" or case.get("dtype") == "i8":
        return "exact"
    # 32-bit sums in another order: 1e-5 of the result's norm, single elements 40 times that of its root mean square
    return {"rel": 1e-5}

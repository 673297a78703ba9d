"""Performance cases: the work a user of this backend has it do, through its public entry points.

Two kinds of caller exist.  A service loads a quantised model once (`CVMAPILoadModel`) and calls `CVMAPIInference` with
host bytes for every request; a plug-in host calls the operators one by one on int32 device tensors.  `listed()` names
representative calls of both, `draw(rng)` gives more of the same ranges.  Every result is an integer: all comparisons
are exact.
"""
import functools
import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.load_package()
from cvm_runtime_amd import graphgen, hipops, runtime  # noqa: E402


def listed():
    return [
        # one image per call: a node that verifies single inferences; ResNet-20 is the smallest graph, pure latency
        {"name": "resnet20 b1", "kind": "model", "net": "resnet20", "batch": 1, "size": 32},
        # a batch of small images
        {"name": "resnet20 b64", "kind": "model", "net": "resnet20", "batch": 64, "size": 32},
        # the common single-image classification request
        {"name": "resnet50 b1", "kind": "model", "net": "resnet50", "batch": 1, "size": 224},
        # the headline configuration
        {"name": "resnet50 b16", "kind": "model", "net": "resnet50", "batch": 16, "size": 224},
        # a service that empties its queue into one call: large, and not a power of two
        {"name": "resnet50 b50", "kind": "model", "net": "resnet50", "batch": 50, "size": 224},
        # the graph with the largest layers and the largest filters
        {"name": "vgg16 b16", "kind": "model", "net": "vgg16", "batch": 16, "size": 224},
        # detector: depthwise layers, heads, get_valid_counts and NMS inside one graph
        {"name": "ssd512 b1", "kind": "model", "net": "ssd", "batch": 1, "size": 512},
        # plug-in host, node by node at the int32 contract: a bottleneck block with pooling and the global sum, one image ...
        {"name": "nodes block b1", "kind": "block", "batch": 1, "mid": 64, "size": 56},
        # ... and a batch
        {"name": "nodes block b16", "kind": "block", "batch": 16, "mid": 64, "size": 56},
        # plug-in host: a depthwise-separable layer on an odd-sized map
        {"name": "nodes separable b4", "kind": "separable", "batch": 4, "channels": 96, "out": 160, "size": 75, "stride": 1},
        # the detector's tail as operators: anchors of SSD-512, the usual top_k
        {"name": "detect top400", "kind": "detect", "batch": 1, "rows": 24564, "top_k": 400, "force": False, "keep": -1},
        # the same with the operator's default top_k (every valid row is a candidate)
        {"name": "detect all", "kind": "detect", "batch": 1, "rows": 24564, "top_k": -1, "force": False, "keep": -1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("resnet20", "resnet50", "resnet50", "vgg16", "ssd", "block", "separable", "detect", "detect"))
    if kind == "resnet20":
        return {"kind": "model", "net": kind, "batch": _log_int(rng, 2, 256), "size": 32}
    if kind == "resnet50":
        return {"kind": "model", "net": kind, "batch": _log_int(rng, 1, 50), "size": rng.randint(160, 224)}
    if kind == "vgg16":
        return {"kind": "model", "net": kind, "batch": _log_int(rng, 1, 16), "size": rng.randint(96, 224)}
    if kind == "ssd":
        return {"kind": "model", "net": kind, "batch": 1, "size": rng.randint(256, 512)}
    if kind == "block":
        mid = rng.choice((64, 128, 256))
        return {"kind": "block", "batch": _log_int(rng, 1, 16), "mid": mid, "size": rng.randint(7, 3584 // mid)}
    if kind == "separable":
        return {"kind": "separable", "batch": _log_int(rng, 1, 8), "channels": rng.randint(24, 256), "out": rng.randint(32, 320),
                "size": rng.randint(7, 96), "stride": rng.choice((1, 1, 2))}
    return {"kind": "detect", "batch": rng.randint(1, 4), "rows": _log_int(rng, 1000, 24564), "top_k": rng.choice((-1, 100, 400, 1000)),
            "force": rng.random() < 0.3, "keep": rng.choice((-1, -1, 100))}


# ------------------------------------------------------------------ models
@functools.lru_cache(maxsize=16)
def _graph(net, batch, size):
    """Graph text, parameter blob, multiply-accumulates per pass, input shape."""
    if net == "resnet20":
        g, heads = graphgen.resnet20_cifar(batch)
    elif net == "resnet50":
        g, heads = graphgen.resnet50(batch, size=size)
    elif net == "vgg16":
        g, heads = graphgen.vgg16(batch, size=size)
    else:
        g, heads = graphgen.ssd_mobilenet(size)
    text, params = g.build(heads)
    out = sum(int(np.prod(g.shape(h))) for h in heads)
    return text, params, g.macs, g.shape((0, 0)), out


_loaded = {}   # the one model in use: a service loads it once and keeps it for all its requests


def _model(case):
    key = (case["net"], case["batch"], case["size"])
    if key not in _loaded:
        _loaded.clear()
        text, params = _graph(*key)[:2]
        _loaded[key] = runtime.HipModel(text, params)
    return _loaded[key]


# ------------------------------------------------------------------ inputs
def _rand(gen, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, dtype=torch.int32, device="cuda", generator=gen)


def _rows(gen, batch, n):
    """Detector rows (id, score, x1, y1, x2, y2): boxes of 16 to 256 pixels around points of a 512-pixel image."""
    dev = "cuda"
    rows = torch.empty((batch, n, 6), dtype=torch.int32, device=dev)
    rows[..., 0] = _rand(gen, (batch, n), 0, 20)
    rows[..., 1] = (torch.randn((batch, n), device=dev, generator=gen) * 30).round().clamp(-127, 127).int()
    centre = torch.rand((batch, n, 2), device=dev, generator=gen) * 512
    half = 8 * torch.exp2(4 * torch.rand((batch, n, 2), device=dev, generator=gen))
    rows[..., 2:4] = (centre - half).clamp(0, 511).int()
    rows[..., 4:6] = (centre + half).clamp(0, 511).int()
    return rows


def prepare(case, seed):
    if case["kind"] == "model":
        # images as the host receives them: int8 bytes over the whole range
        model, shape = _model(case), _graph(case["net"], case["batch"], case["size"])[3]
        data = np.random.default_rng(seed).integers(-127, 128, int(np.prod(shape)), dtype=np.int8)
        kind = np.int32 if runtime.CVMAPIGetOutputTypeSize(model.net) == 4 else np.int8
        return {"kind": "model", "model": model, "data": data.tobytes(), "type": kind}
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    st = {"kind": case["kind"]}
    if case["kind"] == "block":
        n, mid, s = case["batch"], case["mid"], case["size"]
        st["x"] = _rand(gen, (n, 4 * mid, s, s), -127, 127)
        st["w"] = [_rand(gen, v, -127, 127) for v in ((mid, 4 * mid, 1, 1), (mid, mid, 3, 3), (4 * mid, mid, 1, 1))]
        st["b"] = [_rand(gen, (v.shape[0],), -32768, 32768) for v in st["w"]]
        st["shift"] = [graphgen.shift_for(v[0].numel()) for v in st["w"]]
    elif case["kind"] == "separable":
        n, c, oc, s = case["batch"], case["channels"], case["out"], case["size"]
        st["x"] = _rand(gen, (n, c, s, s), -127, 127)
        st["w"] = [_rand(gen, (c, 1, 3, 3), -127, 127), _rand(gen, (oc, c, 1, 1), -127, 127)]
        st["b"] = [_rand(gen, (v.shape[0],), -32768, 32768) for v in st["w"]]
        st["shift"] = [graphgen.shift_for(v[0].numel()) for v in st["w"]]
        st["stride"] = case["stride"]
    else:
        st["x"] = _rows(gen, case["batch"], case["rows"])
        st["top_k"], st["force"], st["keep"] = case["top_k"], case["force"], case["keep"]
    return st


# ------------------------------------------------------------------ one pass
def run(state):
    if state["kind"] == "model":
        return np.frombuffer(state["model"].inference(state["data"]), state["type"])
    x = state["x"]
    if state["kind"] == "block":
        w, b, sh = state["w"], state["b"], state["shift"]
        y = hipops.cvm_right_shift(hipops.relu(hipops.conv2d(x, w[0], b[0])), 8, sh[0])
        y = hipops.cvm_right_shift(hipops.relu(hipops.conv2d(y, w[1], b[1], padding=(1, 1))), 8, sh[1])
        y = hipops.cvm_right_shift(hipops.conv2d(y, w[2], b[2]), 8, sh[2])
        y = hipops.cvm_clip(hipops.cvm_right_shift(hipops.relu(hipops.elemwise("elemwise_add", y, x)), 8, 1), 8)
        return {"out": y, "pooled": hipops.max_pool2d(y, (3, 3), (2, 2), (1, 1)), "sums": hipops.reduce("sum", y, (2, 3))}
    if state["kind"] == "separable":
        w, b, sh = state["w"], state["b"], state["shift"]
        s = (state["stride"], state["stride"])
        y = hipops.conv2d(x, w[0], b[0], s, (1, 1), groups=x.shape[1])
        y = hipops.cvm_right_shift(hipops.relu(y), 8, sh[0])
        y = hipops.conv2d(y, w[1], b[1])
        return hipops.cvm_right_shift(hipops.relu(y), 8, sh[1])
    count, rows = hipops.get_valid_counts(x, 10)
    out = torch.empty_like(rows)
    hipops.non_max_suppression(rows, count, out, 45, state["force"], state["top_k"], max_output_size=state["keep"])
    return {"count": count, "rows": out}


def work(case):
    """Bytes and operations a pass cannot do without: inputs, parameters and outputs once, true multiply-accumulates."""
    if case["kind"] == "model":
        _, params, macs, shape, out = _graph(case["net"], case["batch"], case["size"])
        return {"bytes": float(np.prod(shape)) + len(params) + 4.0 * out, "flops": 2.0 * macs}
    if case["kind"] == "block":
        n, mid, s = case["batch"], case["mid"], case["size"]
        ops = 17 * mid * mid
        half = (s + 1) // 2
        return {"bytes": 4.0 * (n * 4 * mid * (2 * s * s + half * half + 1) + ops + 6 * mid), "flops": 2.0 * n * s * s * ops}
    if case["kind"] == "separable":
        n, c, oc, s = case["batch"], case["channels"], case["out"], case["size"]
        o = (s - 1) // case["stride"] + 1
        return {"bytes": 4.0 * (n * (c * s * s + oc * o * o) + c * (9 + oc) + c + oc), "flops": 2.0 * n * o * o * c * (9 + oc)}
    return {"bytes": 4.0 * (12 * case["batch"] * case["rows"] + case["batch"]), "flops": 0.0}


def tolerance(case):
    return "exact"

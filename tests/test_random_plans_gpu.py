"""Seeded random networks whose tensors have several readers, several heads and lent storage, in every launch form that
the planner chooses between, against the oracle running the graph node by node."""
import json

import numpy as np
import pytest

import oracle.graph as og
from cvm_runtime_amd import graphgen, runtime, synth

pytestmark = pytest.mark.gpu

FORMS = [{}, {"CVM_HIP_RESIDENT": "0"}, {"CVM_HIP_RESIDENT": "1"}, {"CVM_HIP_SEQ": "1"}, {"CVM_HIP_SEQ": "0"}]


def _network(seed):
    rng = np.random.RandomState(seed)
    g = graphgen.GraphBuilder("plans-%d" % seed)
    n, c, hw = (int(rng.choice(v)) for v in ((1, 2, 3, 8, 16), (1, 3, 3, 16, 32, 64), (3, 5, 8, 12, 17)))
    widths = [128, 256, 512] if rng.rand() < 0.4 else [3, 16, 32, 48, 64, 96, 128]
    x = g.var("data", (n, c, hw, hw), 8)
    maps, rows = [x], []
    for _ in range(int(rng.randint(4, 14))):
        cur = maps[-1] if rng.rand() < 0.65 else maps[int(rng.randint(len(maps)))]
        _, cc, h, w = g.shape(cur)
        kind = rng.choice(["conv", "conv", "conv", "whole", "dw", "pair", "pair", "add", "pool", "concat", "abs", "scale", "dense", "sum"])
        stride = int(rng.choice([1, 1, 2])) if h >= 3 else 1
        alike = [t for t in maps if t is not cur and g.shape(t)[2:] == (h, w)]
        other = alike[int(rng.randint(len(alike)))] if alike else None
        if kind == "conv":
            k = int(rng.choice([1, 1, 3]))
            maps.append(g.conv_relu_q(cur, int(rng.choice(widths)), k, stride, k // 2, relu=bool(rng.randint(2))))
        elif kind == "whole" and cc * h * h < 5000:       # a 1x1 result
            maps.append(g.conv_relu_q(cur, int(rng.choice(widths)), h))
        elif kind == "dw" and cc >= 8:
            maps.append(g.conv_relu_q(cur, cc, 3, stride, 1, groups=cc))
        elif kind == "pair":                              # depthwise, then 1x1
            if cc % 32:
                cc = 32 * int(rng.choice([1, 2, 4]))
                maps.append(g.conv_relu_q(cur, cc, 1))
            maps.append(g.conv_relu_q(maps[-1] if g.shape(cur)[1] != cc else cur, cc, 3, stride, 0 if h >= 3 and rng.rand() < 0.4 else 1, groups=cc))
            maps.append(g.conv_relu_q(maps[-1], int(rng.choice([32, 64, 96, 128, 256])), 1))
        elif kind == "add" and other is not None and g.shape(other) == g.shape(cur):
            y = g.add(cur, other)
            maps.append(g.rshift(g.relu(y) if rng.randint(2) else y, 1))
        elif kind == "pool" and h >= 3:
            maps.append(g.max_pool(cur, 3, 2, 1) if rng.randint(2) or h % 2 else g.max_pool(cur, 2, 2))
        elif kind == "concat" and other is not None:
            maps.append(g.concat([cur, other], 1))
        elif kind == "abs":
            maps.append(g.unary("abs", cur))
        elif kind == "scale":
            y, k = g.conv(cur, int(rng.choice(widths)), 1)
            y = g.op("broadcast_mul", [y, g.param("m%d" % g._n, (1,), 3, 3, 3)], {}, [g.shape(y)])[0]
            maps.append(g.rshift(g.relu(y), graphgen.shift_for(k) + 2))
        elif kind == "sum" or (kind == "dense" and cc * h * w <= 30000):
            if kind == "sum":
                cur = g.rshift(g.global_sum(cur)[0], max(1, int(np.ceil(np.log2(h * w)))))
            y = g.flatten(cur)
            for units in (int(rng.choice([10, 33, 64, 128])), int(rng.choice([7, 40])))[:int(rng.randint(1, 3))]:
                y, k = g.dense(y, units)
                y = g.rshift(y, graphgen.shift_for(k))
            rows.append(y)
    if len(maps) == 1:
        maps.append(g.conv_relu_q(x, 16, 1))
    heads = [t for t in maps[1:] + rows if g._eid(t) not in g.consumers or rng.rand() < 0.1][-6:]
    js, pb = g.build([g.reshape(t, (n, 1, int(np.prod(g.shape(t)[1:])))) for t in heads])
    return (_lend(js, rng) if rng.rand() < 0.5 else js), pb, (n, c, hw, hw)


def _lend(js, rng):
    """Storage of tensors that nobody reads any more goes to later results, as a memory-planned graph has it."""
    doc = json.loads(js)
    row, last, sids, kept = doc["node_row_ptr"], {}, [], set()
    for nid, node in enumerate(doc["nodes"]):
        for e in node["inputs"]:
            last[row[e[0]] + e[1]] = nid
    for e in doc["heads"]:
        last[row[e[0]] + e[1]] = len(doc["nodes"])
    for nid, node in enumerate(doc["nodes"]):
        busy = kept | {s for e, s in enumerate(sids) if last.get(e, -1) >= nid}
        free = sorted(set(sids) - busy)
        for _ in range(row[nid], row[nid + 1]):
            if node["op"] != "null" and free and rng.rand() < 0.7:
                sids.append(free.pop(int(rng.randint(len(free)))))
            else:
                sids.append(max(sids, default=-1) + 1)
                if node["op"] == "null" and node["name"] != "data":
                    kept.add(sids[-1])
    doc["attrs"]["storage_id"][1] = sids
    return json.dumps(doc)


@pytest.mark.parametrize("first", range(0, 160, 20))
def test_every_launch_form_of_random_networks(first, dev, monkeypatch):
    for seed in range(first, first + 20):
        js, pb, shape = _network(seed)
        params = graphgen.load_params(pb)
        inputs = [synth.tensor("plans-%d" % seed, "x%d" % i, shape, -127, 127) for i in range(2)]
        wants = [np.concatenate([v.reshape(shape[0], -1) for v in og.run_graph(js, params, x)], axis=1).ravel() for x in inputs]
        for form in FORMS:
            with monkeypatch.context() as env:
                for name, value in form.items():
                    env.setenv(name, value)
                m = runtime.HipModel(js, pb)
            kind = np.int32 if runtime.CVMAPIGetOutputTypeSize(m.net) == 4 else np.int8
            for call in range(4):
                got = np.frombuffer(m.inference(inputs[call % 2].astype(np.int8).tobytes()), kind).astype(np.int32)
                assert np.array_equal(got, wants[call % 2]), "seed %d %s call %d" % (seed, form, call)
            m.close()

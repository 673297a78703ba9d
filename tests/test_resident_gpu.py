"""Layers whose maps stay in LDS, one launch for all of them, against the oracle running the graph node by node."""
import numpy as np
import pytest

import oracle.graph as og
from cvm_runtime_amd import graphgen, runtime, synth

pytestmark = pytest.mark.gpu


def _net(case, batch):
    """A few layers with the forms that a launch tells apart; every case ends in sum and dense."""
    name, c, h, w, widths = case
    g = graphgen.GraphBuilder("resident-" + name)
    x = g.var("data", (batch, c, h, w), 8)
    x = g.conv_relu_q(x, widths[0], 3, 1, 1)
    for i, oc in enumerate(widths[1:]):
        y, k = g.conv(x, oc, 3, 1 + i % 2, 1 + (name == "dilated"), dilation=2 if name == "dilated" else 1)
        if name == "multiply":
            y = g.rshift(g.op("broadcast_mul", [y, g.param("m%d" % i, (1,), 3, 3, 3)], {}, [g.shape(y)])[0], graphgen.shift_for(k) + 2)
        else:
            y = g.rshift(g.relu(y), graphgen.shift_for(k))
        z = g.conv_relu_q(y, oc, 1, relu=False)
        x = g.rshift(g.relu(g.add(z, y)), 1)
        if name == "pooled":
            x = g.max_pool(x, 2, 2) if i % 2 else g.max_pool(x, 3, 2, 1)
    s, _ = g.global_sum(x)
    y, _ = g.dense(g.flatten(g.rshift(s, 4)), 7)
    return g, [y]


CASES = [
    ("tile", 3, 16, 16, (16, 16, 32)),            # whole tiles of 16 pixels in a row
    ("odd", 1, 7, 13, (5, 20, 33)),               # rows, channels and tiles with remainders
    ("small", 3, 4, 3, (16, 48)),                 # fewer tiles than wavefronts
    ("wide", 3, 8, 8, (64, 48, 80)),               # filters of several chunks
    ("dilated", 2, 12, 11, (24, 24, 24)),
    ("multiply", 3, 10, 16, (16, 16, 16)),        # a chain that is no shift and clip
    ("pooled", 3, 18, 22, (16, 24, 40)),
]


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_small_maps_stay_in_lds(case, batch, dev, monkeypatch):
    g, heads = _net(case, batch)
    js, pb = g.build(heads)
    x = synth.tensor("resident-" + case[0], "data", (batch,) + case[1:4], -127, 127).astype(np.int8)
    monkeypatch.setenv("CVM_HIP_RESIDENT", "1")
    m = runtime.HipModel(js, pb)
    steps = m.launch_counts()[0]
    assert steps <= 3, steps          # the packed image, the launch, and at most what its last layer leaves
    got = [np.frombuffer(m.inference(x.tobytes()), np.int32) for _ in range(3)]
    m.run()                           # the same input again, in the staged form
    got.append(np.frombuffer(m.get_output(), np.int32))
    m.close()
    want = og.run_graph(js, graphgen.load_params(pb), x.astype(np.int32))[0].ravel()
    for v in got:
        assert np.array_equal(v, want)


def test_images_in_rounds(dev):
    """More images than compute units: workgroups take a second image."""
    g, heads = _net(CASES[0], 261)
    js, pb = g.build(heads)
    x = synth.tensor("resident-rounds", "data", (261, 3, 16, 16), -127, 127).astype(np.int8)
    m = runtime.HipModel(js, pb)
    got = np.frombuffer(m.inference(x.tobytes()), np.int32).reshape(261, -1)
    m.close()
    for i in (0, 1, 255, 256, 260):
        one, heads1 = _net(CASES[0], 1)
        j1, p1 = one.build(heads1)
        assert np.array_equal(got[i], og.run_graph(j1, graphgen.load_params(p1), x[i:i + 1].astype(np.int32))[0].ravel())


def _check_heads(g, heads, n, cid, monkeypatch):
    js, pb = g.build([g.reshape(t, (n, 1, int(np.prod(g.shape(t)[1:])))) for t in heads])
    params = graphgen.load_params(pb)
    results = []
    for resident in ("1", "0"):
        monkeypatch.setenv("CVM_HIP_RESIDENT", resident)
        m = runtime.HipModel(js, pb)
        results.append(m.launch_counts()[0])
        kind = np.int32 if runtime.CVMAPIGetOutputTypeSize(m.net) == 4 else np.int8
        for i in range(3):
            x = synth.tensor(cid, "data%d" % i, g.shape((0, 0)), -127, 127)
            want = np.concatenate([v.reshape(n, -1) for v in og.run_graph(js, params, x)], axis=1).ravel()
            got = np.frombuffer(m.inference(x.astype(np.int8).tobytes()), kind).astype(np.int32)
            assert np.array_equal(got, want), "resident %s call %d" % (resident, i)
        m.close()
    return results


def test_a_map_that_a_sum_reads_before_a_pool_does(dev, monkeypatch):
    """The launch loads the map where the sum needs it, and the pool behind needs its rows."""
    g = graphgen.GraphBuilder("resident-sum-first")
    x = g.conv_relu_q(g.var("data", (4, 16, 17, 15), 8), 16, 3, 2, 1, groups=16)   # not a layer of such a launch
    s, _ = g.global_sum(x)
    d, k = g.dense(g.flatten(g.rshift(s, 7)), 128)
    d, _ = g.dense(g.rshift(d, graphgen.shift_for(k)), 7)
    y = g.conv_relu_q(g.conv_relu_q(g.max_pool(x, 3, 2, 1), 64, 1, 2), 32, 3, 1, 1)
    launches = _check_heads(g, [y, g.rshift(d, 10)], 4, "resident-sum-first", monkeypatch)
    assert launches[0] < launches[1], launches     # layers in LDS at all


def test_the_image_packed_for_a_convolution_outside_the_launch_is_written(dev, monkeypatch):
    """Two convolutions over the input pack it for themselves; the launch may take the first one and not the second."""
    g = graphgen.GraphBuilder("resident-two-stems")
    x = g.var("data", (16, 1, 3, 3), 8)
    a = g.conv_relu_q(x, 512, 3, 1, 1, relu=False)
    b = g.conv_relu_q(g.conv_relu_q(x, 256, 3, 2, 1), 512, 1)      # 512 x 256: the filter does not fit beside the rest
    b = g.conv_relu_q(g.conv_relu_q(b, 256, 1), 256, 3, 1, 1, groups=256)
    _check_heads(g, [a, b], 16, "resident-two-stems", monkeypatch)


@pytest.mark.parametrize("h,w,channels,pad,batch", [
    (16, 32, (16, 16), 1, 2),        # two tiles of a row and the two below
    (18, 64, (12, 16), 1, 1),        # several of these in a row; channels past the last
    (6, 96, (16, 9), 1, 1),
    (32, 16, (16, 16), 1, 2),        # four rows of a map one tile wide
    (34, 16, (16, 16), 1, 1),        # not a multiple of four: tiles on their own
    (18, 34, (16, 16), 0, 1),        # a window that begins inside the map
    (16, 32, (16, 32, 16), 1, 1),
    (64, 64, (16, 16, 16), 1, 100),  # images past 1 MiB: the kernel reads the copy on the device
])
def test_rows_that_share_operands(h, w, channels, pad, batch, dev, monkeypatch):
    def net(n):
        g = graphgen.GraphBuilder("resident-rows")
        x = g.conv_relu_q(g.var("data", (n, 3, h, w), 8), channels[0], 3, 1 + h // 64, 1)
        for oc in channels[1:]:
            y = g.conv_relu_q(x, oc, 3, 1, pad)
            z = g.conv_relu_q(y, oc, 3, 1, 1, relu=False)
            x = g.rshift(g.relu(g.add(z, y)), 1)
        s, _ = g.global_sum(x)
        y, _ = g.dense(g.flatten(g.rshift(s, 6)), 5)
        return g.build([y])

    js, pb = net(batch)
    x = synth.tensor("resident-rows", "data", (batch, 3, h, w), -127, 127).astype(np.int8)
    monkeypatch.setenv("CVM_HIP_RESIDENT", "1")
    m = runtime.HipModel(js, pb)
    assert m.launch_counts()[0] <= 3
    got = [np.frombuffer(m.inference(x.tobytes()), np.int32).reshape(batch, -1) for _ in range(2)]
    m.close()
    j1, p1 = net(1)
    p1 = graphgen.load_params(p1)
    for i in {0, 1 % batch, batch // 2, batch - 1}:
        want = og.run_graph(j1, p1, x[i:i + 1].astype(np.int32))[0].ravel()
        for v in got:
            assert np.array_equal(v[i], want), i

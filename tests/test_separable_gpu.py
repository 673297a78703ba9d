"""Depthwise and 1x1 convolution in one launch, against the oracle running the graph node by node."""
import ctypes
import json

import numpy as np
import pytest

import oracle.graph as og
from cvm_runtime_amd import check, graphgen, lib, runtime, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,h,w,oc,stride,pad", [
    (1, 32, 67, 61, 32, 1, 1),       # one channel tile: 256 pixels to a workgroup, ends inside one
    (2, 64, 40, 40, 64, 2, 1),
    (1, 96, 33, 50, 160, 1, 0),      # no padding; channel tiles that do not fill the last workgroup
    (3, 128, 23, 30, 128, 1, 1),
    (1, 512, 29, 31, 512, 1, 1),     # the depthwise tile computed by two workgroups
    (1, 288, 30, 30, 320, 2, 2),     # padding wider than the filter needs, a second group of two channel tiles
    (1, 512, 17, 18, 1024, 2, 1),    # filter requested in two rounds, four groups
])
@pytest.mark.parametrize("multiply", [False, True])
def test_depthwise_and_pointwise_in_one_launch(n, c, h, w, oc, stride, pad, multiply, dev, monkeypatch):
    g = graphgen.GraphBuilder("separable-%d-%d" % (c, oc))
    x = g.var("data", (n, c, h, w), 8)
    y, k = g.conv(x, c, 3, stride, pad, groups=c)
    if multiply:   # a chain that is no clamp and shift
        y = g.op("broadcast_mul", [y, g.param("m", (1,), 3, 3, 3)], {}, [g.shape(y)])[0]
    y = g.rshift(g.relu(y), graphgen.shift_for(k) + 2 * multiply)
    z, k = g.conv(y, oc, 1)
    z = g.conv_relu_q(g.rshift(z, graphgen.shift_for(k)), 40, 1)   # reads it as int8
    js, pb = g.build([z])
    data = synth.tensor("separable", "data%d" % c, (n, c, h, w), -127, 127)
    monkeypatch.setenv("CVM_HIP_RESIDENT", "1")
    m = runtime.HipModel(js, pb)
    counts = [m.launch_counts()[0]]
    got = np.frombuffer(m.inference(data.astype(np.int8).tobytes()), np.int8 if m.output_length == int(np.prod(g.shape(z))) else np.int32)
    m.close()
    monkeypatch.setenv("CVM_HIP_SEPARABLE", "0")
    m = runtime.HipModel(js, pb)
    counts.append(m.launch_counts()[0])
    m.close()
    assert counts[0] == counts[1] - 1, counts
    assert np.array_equal(got.astype(np.int32), og.run_graph(js, graphgen.load_params(pb), data.astype(np.int32))[0].ravel())


def test_a_depthwise_result_that_a_dense_layer_reads_too_is_written(dev, monkeypatch):
    """flatten of a 1x1 map shares the map's memory under another entry: the 1x1 convolution is not its only reader."""
    g = graphgen.GraphBuilder("separable-flatten")
    x = g.var("data", (2, 512, 3, 3), 8)
    y = g.conv_relu_q(x, 512, 3, 1, 0, groups=512)
    z = g.conv_relu_q(g.conv_relu_q(y, 512, 1), 40, 1)
    d, _ = g.dense(g.flatten(y), 24)
    js, pb = g.build([g.reshape(z, (2, 1, 40)), g.reshape(g.rshift(d, 9), (2, 1, 24))])
    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")    # the layers behind would do without the tensor's memory
    counts = []
    for separable in ("1", "0"):
        monkeypatch.setenv("CVM_HIP_SEPARABLE", separable)
        m = runtime.HipModel(js, pb)
        counts.append(m.launch_counts()[0])
        for i in range(3):
            data = synth.tensor("separable-flatten", "data%d" % i, (2, 512, 3, 3), -127, 127)
            want = og.run_graph(js, graphgen.load_params(pb), data.astype(np.int32))
            got = np.frombuffer(m.inference(data.astype(np.int8).tobytes()), np.int8).astype(np.int32)
            assert np.array_equal(got, np.concatenate([v.reshape(2, -1) for v in want], axis=1).ravel())
        m.close()
    assert counts[0] == counts[1], counts


@pytest.mark.parametrize("n,c,hw,oc,fused", [
    (3, 96, 128, 96, True), (4, 96, 128, 96, False),          # 48 K and 64 K pixels, three channel tiles
    (1, 32, 128, 128, True), (4, 32, 128, 128, False),        # four times the channels
    (8, 64, 128, 128, True), (9, 64, 128, 128, False),        # twice: 128 K pixels and more
    (4, 32, 512, 32, True), (5, 32, 512, 32, False),          # as many: 1 M pixels and more
])
def test_pairs_of_many_pixels_stay_two_launches(n, c, hw, oc, fused, dev, monkeypatch):
    g = graphgen.GraphBuilder("separable-rule-%d-%d" % (c, oc))
    z = g.conv_relu_q(g.conv_relu_q(g.var("data", (n, c, hw, hw), 8), c, 3, 1, 1, groups=c), oc, 1)
    js, pb = g.build([g.conv_relu_q(z, 40, 1)])
    monkeypatch.setenv("CVM_HIP_RESIDENT", "1")
    counts = []
    for separable in ("1", "0"):
        monkeypatch.setenv("CVM_HIP_SEPARABLE", separable)
        m = runtime.HipModel(js, pb)
        counts.append(m.launch_counts()[0])
        m.close()
    assert counts[1] - counts[0] == fused, counts


@pytest.mark.parametrize("n,c,h,w,pool", [
    (10, 3, 64, 128, True),       # whole patches of 32 x 16
    (9, 1, 62, 130, True),        # patches that end outside
    (9, 3, 61, 131, False),
    (8, 4, 40, 250, True),        # outside on both sides
    (8, 3, 39, 250, False),
    (600, 3, 16, 30, False),      # several patches to a workgroup
    (7, 3, 64, 128, True),        # too few
])
def test_first_two_layers_of_a_vgg(n, c, h, w, pool, dev, monkeypatch):
    def net(k):
        g = graphgen.GraphBuilder("stem-conv-%d-%d" % (c, w))
        x = g.conv_relu_q(g.var("data", (k, c, h, w), 8), 64, 3, 1, 1)
        y = g.conv_relu_q(x, 64, 3, 1, 1)
        return g.build([g.conv_relu_q(g.max_pool(y, 2, 2) if pool else y, 8, 1)])

    js, pb = net(n)
    x = synth.tensor("stem-conv", "x%d" % w, (n, c, h, w), -128, 127)
    out, launches = [], []
    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")
    for pair in ("1", "0"):
        monkeypatch.setenv("CVM_HIP_SEPARABLE", pair)
        m = runtime.HipModel(js, pb)
        launches.append(m.launch_counts()[0])
        for _ in range(4):   # eager, capture, replays
            out.append(np.frombuffer(m.inference(x.astype(np.int8).tobytes()), np.int8).reshape(n, -1))
        m.close()
    assert launches[1] - launches[0] == (0 if n == 7 else 1), launches
    j1, p1 = net(1)
    p1 = graphgen.load_params(p1)
    for i in (0, n - 1):
        want = og.run_graph(j1, p1, np.clip(x[i:i + 1], -127, 127))[0].ravel()
        for v in out:
            assert np.array_equal(v[i], want), i
    for v in out[1:]:
        assert np.array_equal(v, out[0])


@pytest.mark.parametrize("n,h,w,pool,patches", [
    (5, 130, 170, True, "64 x 8"),      # 270 patches of 32 x 16, 255 of 64 x 8: one round of workgroups instead of two
    (5, 130, 170, False, "64 x 8"),
    (14, 66, 122, True, "64 x 8"),      # 280 and 252; patches that end outside on both sides
    (8, 130, 170, True, "32 x 16"),     # 432 and 408: two rounds either way
    (35, 36, 180, False, "32 x 16"),    # 630 and 525: three
    (29, 66, 128, True, "32 x 16"),
])
def test_patches_of_the_first_two_layers(n, h, w, pool, patches, dev, monkeypatch):
    def net(k):
        g = graphgen.GraphBuilder("stem-patch-%d" % w)
        y = g.conv_relu_q(g.conv_relu_q(g.var("data", (k, 3, h, w), 8), 64, 3, 1, 1), 64, 3, 1, 1)
        return g.build([g.conv_relu_q(g.max_pool(y, 2, 2) if pool else y, 8, 1)])

    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")
    js, pb = net(n)
    x = synth.tensor("stem-patch", "x%d" % w, (n, 3, h, w), -127, 127)
    out = []
    for pair in ("1", "0"):
        monkeypatch.setenv("CVM_HIP_SEPARABLE", pair)
        m = runtime.HipModel(js, pb)
        check(lib().cvmhip_kernel_timing_begin())
        out.append(np.frombuffer(m.inference(x.astype(np.int8).tobytes()), np.int8).reshape(n, -1))
        buf = ctypes.create_string_buffer(1 << 16)
        check(lib().cvmhip_kernel_timing_end_launches(buf, len(buf)))
        launches = [e["desc"] for e in json.loads(buf.value.decode()) if e["desc"].startswith("3x3/1 3->64 and")]
        assert [d.split("patches of ")[1] for d in launches] == ([patches] if pair == "1" else [])
        m.close()
    assert np.array_equal(out[0], out[1])
    j1, p1 = net(1)
    for i in (0, n - 1):
        assert np.array_equal(out[0][i], og.run_graph(j1, graphgen.load_params(p1), x[i:i + 1])[0].ravel()), i

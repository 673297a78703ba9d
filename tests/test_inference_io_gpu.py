"""The two ends of CVMAPIInference: the caller's bytes through the pinned buffer (pieces, odd sizes, the clamp) into the
row-window or the plain layout, and the outputs with their ticket back -- against the oracle's graph executor."""
import json

import numpy as np
import pytest

import oracle.graph as og
from cvm_runtime_amd import graphgen, runtime, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,h,w,k,stride,precision,second_reader", [
    (1, 1, 1, 1, 1, 1, 8, False),       # one byte in
    (1, 3, 5, 7, 3, 1, 6, False),       # rows that are not whole stores, values beyond the input's precision
    (2, 4, 17, 13, 7, 2, 8, False),
    (1, 3, 9, 33, 5, 2, 7, True),       # a second reader of the input: it exists as int32 too
    (3, 32, 6, 6, 3, 1, 8, False),      # not a row-window layer
    (7, 3, 224, 225, 3, 2, 8, False),   # several pieces, the last one ragged
])
def test_inference_ends(n, c, h, w, k, stride, precision, second_reader, dev):
    g = graphgen.GraphBuilder("io-%d-%d-%d" % (n, c, w))
    x = g.var("data", (n, c, h, w), precision)
    heads = [g.conv_relu_q(x, 32, k, stride, k // 2)]
    if second_reader:
        heads = [g.reshape(heads[0], (n, 1, int(np.prod(g.shape(heads[0])[1:])))), g.reshape(g.clip8(x), (n, 1, c * h * w))]
    js, pb = g.build(heads)
    model = runtime.HipModel(js, pb)
    params = graphgen.load_params(pb)
    top = (1 << (precision - 1)) - 1
    for call in range(3):   # eager, capture, replay, each on another input
        data = synth.tensor("io", "x%d" % call, (n, c, h, w), -128, 127)
        want = og.run_graph(js, params, np.clip(data, -top, top))
        want = want[0].ravel() if len(want) == 1 else np.concatenate([v.reshape(n, -1) for v in want], axis=1).ravel()
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want), "call %d" % call
    model.close()


@pytest.mark.parametrize("patience", ["", "0"])   # the packing launch follows the host's copy; it gives up at once and the call is run again
@pytest.mark.parametrize("n,c,h,w,k,stride,precision", [
    (3, 3, 224, 225, 3, 2, 6),        # rows that begin anywhere in a granule, several chunks to an image, the clamp
    (1, 3, 511, 513, 7, 1, 8),        # one image
    (300, 1, 31, 33, 5, 2, 8),        # many images to a chunk's worth of bytes
    (2, 4, 5, 9001, 3, 1, 8),         # a band of one row
    (5, 3, 260, 90, 3, 1, 8),
])
def test_packing_follows_the_copy(n, c, h, w, k, stride, precision, patience, dev, monkeypatch):
    if patience:
        monkeypatch.setenv("CVM_HIP_GATE_US", patience)
    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")
    g = graphgen.GraphBuilder("io-gate-%d-%d-%d" % (n, c, w))
    x = g.var("data", (n, c, h, w), precision)
    js, pb = g.build([g.conv_relu_q(x, 8, k, stride, k // 2)])
    model = runtime.HipModel(js, pb)
    params = graphgen.load_params(pb)
    top = (1 << (precision - 1)) - 1
    for call in range(5):   # eager, capture, replays; each on another input
        data = synth.tensor("io-gate", "x%d" % call, (n, c, h, w), -128, 127)
        want = og.run_graph(js, params, np.clip(data, -top, top))[0].ravel()
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want), "call %d" % call
        if call == 3:   # the same input again, as a run of its own
            model.run()
            assert np.array_equal(np.frombuffer(model.get_output(), np.int8).astype(np.int32), want)
    model.close()


@pytest.mark.parametrize("patience,calls,told", [("0", 67, 1), ("0", 68, 2), ("0,500000", 200, 1)])
def test_packing_is_tried_again(patience, calls, told, dev, monkeypatch, capfd):
    """A packing launch that gives up says so; 64 calls later the form is taken again, and stays if that one does not."""
    monkeypatch.setenv("CVM_HIP_GATE_US", patience)
    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")
    g = graphgen.GraphBuilder("io-again")
    js, pb = g.build([g.conv_relu_q(g.var("data", (1, 3, 300, 300), 8), 8, 3, 2, 1)])
    model = runtime.HipModel(js, pb)
    params = graphgen.load_params(pb)
    inputs = [synth.tensor("io-again", str(i), (1, 3, 300, 300), -127, 127) for i in range(3)]
    want = [og.run_graph(js, params, v)[0].ravel() for v in inputs]
    for i in range(calls):   # the third is the first with a packing launch
        got = np.frombuffer(model.inference(inputs[i % 3].astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want[i % 3]), i
    model.close()
    assert capfd.readouterr().err.count("the host was kept from copying") == told


def test_many_calls_in_a_row(dev):
    """Past the 64 calls after which the stream itself is waited for; outputs of several kilobytes."""
    g, heads = graphgen.conv_op_graph(n=1, c=32, h=9, w=9, oc=40)
    js, pb = g.build(heads)
    model = runtime.HipModel(js, pb)
    params = graphgen.load_params(pb)
    inputs = [synth.tensor("io-many", str(i), (1, 32, 9, 9), -127, 127) for i in range(3)]
    want = [og.run_graph(js, params, v)[0].ravel() for v in inputs]
    for i in range(140):
        got = np.frombuffer(model.inference(inputs[i % 3].astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want[i % 3]), i
    model.close()


@pytest.mark.parametrize("resident", ["0", "1"])
def test_the_storage_of_the_input_lent_to_a_later_tensor(resident, dev, monkeypatch):
    """A second row-window convolution over a tensor in the place that `data` had takes that tensor, not the input."""
    g = graphgen.GraphBuilder("io-lent")
    x = g.var("data", (2, 3, 12, 12), 8)
    y = g.conv_relu_q(x, 3, 3, 1, 1, relu=False)
    t = g.unary("abs", y)
    z = g.conv_relu_q(t, 32, 3, 1, 1)
    js, pb = g.build([z])
    doc = json.loads(js)
    sid = doc["attrs"]["storage_id"][1]
    sid[g._eid(t)] = sid[g._eid(x)]
    js = json.dumps(doc)
    monkeypatch.setenv("CVM_HIP_RESIDENT", resident)
    model = runtime.HipModel(js, pb)
    for call in range(3):
        data = synth.tensor("io-lent", "x%d" % call, (2, 3, 12, 12), -127, 127)
        want = og.run_graph(js, graphgen.load_params(pb), data)[0].ravel()
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want), "call %d" % call
    model.close()

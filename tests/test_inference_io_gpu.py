"""The two ends of CVMAPIInference: the caller's bytes through the pinned buffer (pieces, odd sizes, the clamp) into the
row-window or the plain layout, and the outputs with their ticket back -- against the oracle's graph executor."""
import ctypes
import json

import numpy as np
import pytest
import torch

import oracle.graph as og
from cvm_runtime_amd import check, graphgen, lib, runtime, synth

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


@pytest.mark.parametrize("words", [
    [1023], [1024], [1025], [1024 * 3 + 2],
    [1024 * 300 + 5],                # more pieces than the workgroups load at a time
    [70000, 0, 5, 1024 * 65],        # one array without a table among others
])
def test_export_in_pieces(words, dev):
    """Pieces of equal words are told, others written; also where only the first or the last word of one differs."""
    piece, L, align = 1024, lib(), lambda n: (n + 63) // 64 * 64
    arrays = []
    for k, n in enumerate(words):
        a = np.repeat(synth.tensor("pieces", "v%d" % k, ((n + piece - 1) // piece,), -3, 3).astype(np.int32), piece)[:n].copy()
        a[piece * 2::piece * 7] += 1
        a[piece - 1::piece * 5] -= 1
        arrays.append(a)
    src = [torch.from_numpy(a).to(dev) if a.size else torch.zeros(4, dtype=torch.int32, device=dev) for a in arrays]
    tables = [None if k == 1 else n // piece for k, n in enumerate(words)]
    host = ctypes.c_void_p()
    total = 64 + sum(align(n * 4 + 16) + align((t or 0) * 8 + 8) for n, t in zip(words, tables))
    check(L.cvmhip_host_alloc(ctypes.byref(host), ctypes.c_size_t(total)))
    raw = np.ctypeslib.as_array((ctypes.c_uint8 * total).from_address(host.value))
    raw[:64] = 0
    raw[64:] = 0x5a
    at, dst, tab = 64, [], []
    for n, t in zip(words, tables):
        dst.append(at)
        at += align(n * 4 + 16)
        tab.append(None if t is None else at)
        at += align((t or 0) * 8 + 8)
    counter = torch.zeros(2, dtype=torch.int32, device=dev)
    K, vp = len(words), ctypes.c_void_p
    stream = vp(torch.cuda.current_stream().cuda_stream)
    for ticket in (1, 2):
        check(L.cvmhip_export_pieces((vp * K)(*[s.data_ptr() for s in src]), (vp * K)(*[host.value + d for d in dst]),
                                     (vp * K)(*[t and host.value + t for t in tab]), (ctypes.c_int64 * K)(*words), K, None, None,
                                     vp(counter.data_ptr()), host, stream))
        check(L.cvmhip_export_wait(host, ctypes.c_uint32(ticket), stream))
    for k, a in enumerate(arrays):
        got = raw[dst[k]:dst[k] + a.size * 4].view(np.int32).copy()
        assert np.all(raw[dst[k] + a.size * 4:dst[k] + align(a.size * 4 + 16)] == 0x5a)
        if tab[k] is not None:
            t = raw[tab[k]:tab[k] + tables[k] * 8].view(np.uint64)
            assert np.all(raw[tab[k] + tables[k] * 8:tab[k] + tables[k] * 8 + 8] == 0x5a)
            for c in range(tables[k]):
                here = a[c * piece:(c + 1) * piece]
                assert bool(t[c] >> np.uint64(32)) == bool(np.all(here == here[0])), c
                if t[c] >> np.uint64(32):
                    got[c * piece:(c + 1) * piece] = np.uint32(t[c] & np.uint64(0xffffffff)).astype(np.int32)
        assert np.array_equal(got, a), k
    torch.cuda.synchronize()
    check(L.cvmhip_host_free(host))


@pytest.mark.parametrize("heads,postprocess", [(1, None), (2, None), (1, "argmax")])
def test_large_outputs_with_equal_pieces(heads, postprocess, dev):
    """An int32 output of several pieces from inputs that are partly zero: read whole, beside another head, by argmax."""
    g = graphgen.GraphBuilder("io-pieces-%d" % heads)
    x = g.var("data", (1, 3, 132, 132), 8)
    y, _ = g.conv(x, 8, 3, 1, 1, bias=False)
    out = [g.reshape(y, (1, 1, 8 * 132 * 132))]
    if heads == 2:
        out.append(g.reshape(g.relu(y), (1, 1, 8 * 132 * 132)))
    if postprocess:
        out = [y]
    js, pb = g.build(out, postprocess=postprocess)
    model = runtime.HipModel(js, pb)
    params = graphgen.load_params(pb)
    for call in range(4):
        data = synth.tensor("io-pieces", "x%d" % call, (1, 3, 132, 132), -127, 127)
        data[:, :, 30 * call:] = 0
        want = og.run_graph(js, params, data)
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), np.int32)
        if postprocess:
            rows = 8 * 132
            flat = want[0].reshape(rows, 132).ravel().astype(np.int8)
            best = []
            for i in range(0, rows, 132):   # the reference's loop: its row cursor advances by a row's length
                m = 0
                for j in range(i, i + 132):
                    if flat[j] > flat[i + m]:
                        m = j - i
                best.append(m)
            got = got[:len(best)]   # (what is behind them nobody writes)
            assert np.array_equal(got, best), "call %d" % call
        else:
            assert np.array_equal(got, np.concatenate([v.ravel() for v in want])), "call %d" % call
        model.run()
        assert np.array_equal(np.frombuffer(model.get_output(), np.int32)[:got.size], got), "call %d" % call
    model.close()


@pytest.mark.parametrize("narrow", [True, False])
def test_pieces_that_are_equal_in_one_call_and_not_in_the_next(narrow, dev):
    """Words of the call before lie in the pinned buffer where a piece was told: as int8, which is read from there, and as int32; runs of more than 65 536 words."""
    g = graphgen.GraphBuilder("io-turns-%d" % narrow)
    x = g.var("data", (1, 3, 132, 140), 8)
    y, k = g.conv(x, 10, 3, 1, 1, bias=False)
    js, pb = g.build([g.reshape(g.rshift(y, graphgen.shift_for(k)) if narrow else y, (1, 1, 10 * 132 * 140))])
    model = runtime.HipModel(js, pb)
    kind = np.int8 if narrow else np.int32
    assert runtime.CVMAPIGetOutputTypeSize(model.net) == kind().itemsize
    params = graphgen.load_params(pb)
    for call, zero in enumerate([slice(0, 0), slice(0, 132), slice(40, 90), slice(0, 60), slice(0, 0), slice(100, 132)]):
        data = synth.tensor("io-turns", "x%d" % call, (1, 3, 132, 140), -127, 127)
        data[:, :, zero] = 0
        want = og.run_graph(js, params, data)[0].ravel()
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), kind)
        assert np.array_equal(got.astype(np.int32), want), "call %d" % call
        model.run()
        assert np.array_equal(np.frombuffer(model.get_output(), kind), got), "call %d" % call
    model.close()

"""3x3 convolution over many channels of few pixels: every tile at its edges, both strides, the fused pool, against the oracle
and against the wavefront kernel; the lines of the dispatch."""
import ctypes
import json

import numpy as np
import pytest
import torch

import oracle
import oracle.graph as og
from cvm_runtime_amd import check, graphgen, hipops, lib, runtime, synth

pytestmark = pytest.mark.gpu


def T(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(dev)


def clamp_shift(lo, hi, shift):
    c = hipops.Chain()
    c.count = 1
    c.stage[0] = hipops.Stage(5, 0, shift, lo, hi)
    return c


def kernel_of(run):
    lib().cvmhip_kernel_timing_begin()
    out = run()
    torch.cuda.synchronize()
    buf = ctypes.create_string_buffer(1 << 16)
    check(lib().cvmhip_kernel_timing_end_launches(buf, len(buf)))
    return out, str(json.loads(buf.value.decode())[-1])


@pytest.mark.parametrize("n,ic,h,w,oc,stride,pool,lo,hi,shift", [
    (1, 512, 1, 1, 64, 1, False, -508, 508, 2),      # one pixel, all its neighbours padding
    (1, 512, 7, 7, 512, 1, False, 0, 2047, 4),       # a ResNet's last stage
    (1, 1024, 13, 15, 128, 2, False, -128, 127, 0),  # two shares of K to a wavefront, odd extents
    (2, 512, 8, 6, 64, 1, True, -2048, 2047, 4),
    (1, 256, 5, 9, 64, 1, False, -127, 127, 0),      # taps dealt to wavefronts
    (2, 128, 7, 4, 64, 2, False, -127, 127, 0),
])
@pytest.mark.parametrize("bias", [False, True])
def test_against_the_oracle(n, ic, h, w, oc, stride, pool, lo, hi, shift, bias, dev):
    cid = "run-%d-%d-%d" % (n, ic, h)
    x = synth.tensor(cid, "x", (n, ic, h, w), -127, 127)
    wt = synth.tensor(cid, "w", (oc, ic, 3, 3), -127, 127)
    b = synth.tensor(cid, "b", (oc,), -2**31, 2**31 - 1) if bias else None
    v = oracle.conv2d(x, wt, np.zeros(oc, np.int32), (stride, stride), (1, 1), (1, 1), 1)
    if bias:
        v = (v.astype(np.int64) + b.reshape(1, -1, 1, 1)).astype(np.int32)   # (wraps)
    ref = np.clip(v, lo, hi) >> shift
    if pool:
        ref = oracle.max_pool2d(ref, (2, 2), (2, 2), (0, 0), False)
    oh, ow = ref.shape[2:]
    chain = clamp_shift(lo, hi, shift)
    xp, wp = hipops.pack_act_i8(T(x, dev)), hipops.pack_weights(T(wt, dev))
    bt = T(b, dev) if bias else None

    def run():
        if pool:
            return hipops.conv2d_pool2_i8(xp, n, ic, h, w, wp, oc, 3, 3, bt, chain, padding=(1, 1))
        return hipops.conv2d_i8(xp, n, ic, h, w, wp, oc, 3, 3, bt, chain, strides=(stride, stride), padding=(1, 1))
    got, kernel = kernel_of(run)
    assert "k_conv_run" in kernel
    got = hipops.unpack_act_i8(got, n, oc, oh, ow)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("n,ic,h,w,oc,stride,pool,takes", [
    (1, 512, 7, 7, 512, 1, False, True),        # 16 x 16
    (3, 512, 7, 7, 512, 1, False, True),        # 16 channels x 32 pixels
    (6, 512, 7, 7, 512, 1, False, True),        # 32 x 32
    (16, 512, 7, 7, 512, 1, False, True),       # 32 x 64
    (23, 512, 7, 7, 512, 1, False, True),       # 64 x 64
    (1, 512, 14, 14, 512, 2, False, True),
    (4, 512, 13, 15, 512, 2, False, True),
    (16, 512, 14, 14, 512, 2, False, True),
    (1, 512, 14, 14, 512, 1, True, True),       # the pool's tiles
    (3, 512, 14, 14, 512, 1, True, True),
    (6, 512, 14, 14, 512, 1, True, True),
    (16, 512, 14, 14, 512, 1, True, True),
    (2, 1536, 5, 3, 192, 1, False, True),
    (50, 512, 14, 14, 512, 2, False, False),    # a run of more pixels than a wavefront's LDS holds
    (50, 512, 7, 7, 512, 1, False, False),      # 312 tiles of 64 x 64
    (1, 256, 16, 16, 512, 2, False, True),      # fewer channels: two or four wavefronts to 64 of them, each with some of the taps
    (2, 256, 9, 5, 128, 1, False, True),
    (5, 256, 9, 10, 256, 1, False, True),
    (7, 768, 9, 10, 256, 1, False, True),
    (12, 256, 9, 10, 256, 1, False, True),
    (1, 128, 8, 8, 256, 2, False, True),
    (1, 128, 3, 2, 64, 1, False, True),
    (5, 128, 9, 10, 256, 1, False, True),
    (7, 384, 9, 10, 256, 1, False, True),
    (12, 128, 9, 10, 256, 1, False, False),
    (2, 256, 14, 14, 256, 1, True, False),
    (16, 64, 7, 7, 256, 1, False, False),
    (1, 512, 7, 7, 96, 1, False, False),        # channels that are not whole groups of 64
])
def test_tiles_and_lines(n, ic, h, w, oc, stride, pool, takes, dev, monkeypatch):
    gen = torch.Generator(device=dev)
    gen.manual_seed(n * ic + h)
    xp = hipops.pack_act_i8(torch.randint(-127, 128, (n, ic, h, w), dtype=torch.int32, device=dev, generator=gen))
    wp = hipops.pack_weights(torch.randint(-127, 128, (oc, ic, 3, 3), dtype=torch.int32, device=dev, generator=gen))
    bt = torch.randint(-100000, 100000, (oc,), dtype=torch.int32, device=dev, generator=gen)
    chain = clamp_shift(0, 127 << 12, 12)

    def run():
        if pool:
            return hipops.conv2d_pool2_i8(xp, n, ic, h, w, wp, oc, 3, 3, bt, chain, padding=(1, 1))
        return hipops.conv2d_i8(xp, n, ic, h, w, wp, oc, 3, 3, bt, chain, strides=(stride, stride), padding=(1, 1))
    out, kernel = kernel_of(run)
    assert ("k_conv_run" in kernel) == takes, kernel
    monkeypatch.setenv("CVM_HIP_CONV", "wave")
    want, kernel = kernel_of(run)
    assert "k_conv_run" not in kernel
    assert torch.equal(out, want)


def test_beside_a_projection(dev, monkeypatch):
    """Two layers of one tensor that could share a launch: the 3x3 one keeps its own kernel."""
    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")
    monkeypatch.setenv("CVM_HIP_SEQ", "0")
    g = graphgen.GraphBuilder("run-pair")
    a = g.conv_relu_q(g.var("data", (1, 64, 14, 14), 8), 512, 1)
    b, c = g.conv_relu_q(a, 512, 3, 2, 1), g.conv_relu_q(a, 512, 1, 2, relu=False)
    js, pb = g.build([g.clip8(g.relu(g.add(g.conv_relu_q(b, 512, 1, relu=False), c)))])
    model = runtime.HipModel(js, pb)
    data = synth.tensor("run-pair", "x", (1, 64, 14, 14), -127, 127)
    want = og.run_graph(js, graphgen.load_params(pb), data)[0].ravel()
    for call in range(3):
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want), call
    lib().cvmhip_kernel_timing_begin()
    model.run()
    torch.cuda.synchronize()
    buf = ctypes.create_string_buffer(1 << 16)
    check(lib().cvmhip_kernel_timing_end_launches(buf, len(buf)))
    assert sum("k_conv_run" in str(launch) for launch in json.loads(buf.value.decode())) == 1
    model.close()


@pytest.mark.parametrize("n,c,hw,oc,stride,twice,shared", [
    (2, 128, 28, 128, 1, True, True),        # 200 workgroups in the group
    (4, 128, 28, 256, 2, False, True),
    (4, 256, 14, 256, 1, True, True),        # 208
    (8, 256, 14, 256, 1, True, False),       # 400: more than one to a compute unit
    (8, 256, 14, 256, 1, False, True),       # 232
    (2, 512, 7, 512, 1, True, False),        # the smallest tile over 512 channels
    (3, 512, 7, 512, 1, True, True),         # 96
    (10, 512, 7, 512, 1, True, True),        # 256
    (12, 512, 7, 512, 1, True, False),       # 320
])
def test_which_layers_share_a_launch(n, c, hw, oc, stride, twice, shared, dev, monkeypatch):
    """Two layers of one tensor, a 3x3 one and another or a 1x1 one beside it."""
    monkeypatch.setenv("CVM_HIP_RESIDENT", "0")
    monkeypatch.setenv("CVM_HIP_SEQ", "0")
    g = graphgen.GraphBuilder("share-%d-%d-%d" % (n, c, stride))
    x = g.conv_relu_q(g.var("data", (n, 32, hw, hw), 8), c, 1)
    a, b = g.conv_relu_q(x, oc, 3, stride, 1), g.conv_relu_q(x, oc, 3 if twice else 1, stride, 1 if twice else 0)
    js, pb = g.build([g.concat([g.conv_relu_q(a, 32, 1), g.conv_relu_q(b, 32, 1)], 1)])
    model = runtime.HipModel(js, pb)
    data = synth.tensor("share", "x%d" % (n * c), (n, 32, hw, hw), -127, 127)
    want = og.run_graph(js, graphgen.load_params(pb), data)[0].ravel()
    for call in range(3):
        got = np.frombuffer(model.inference(data.astype(np.int8).tobytes()), np.int8).astype(np.int32)
        assert np.array_equal(got, want), call
    lib().cvmhip_kernel_timing_begin()
    model.run()
    torch.cuda.synchronize()
    buf = ctypes.create_string_buffer(1 << 16)
    check(lib().cvmhip_kernel_timing_end_launches(buf, len(buf)))
    assert sum("k_conv_run" in str(launch) for launch in json.loads(buf.value.decode())) == (0 if shared else 1 + twice)
    model.close()


@pytest.mark.parametrize("n,ic,h,w,oc,stride,pool,takes", [
    (3, 384, 41, 41, 128, 2, False, False),     # 1 196 bytes of a channel to a workgroup
    (1, 384, 36, 35, 512, 2, False, False),
    (12, 384, 15, 15, 256, 2, False, True),     # 836, 768 pixels
    (1, 896, 37, 37, 64, 1, False, False),      # 1 369 pixels
    (16, 256, 25, 25, 128, 2, False, False),    # 2 704 pixels, 886 bytes
    (1, 256, 45, 45, 128, 1, False, True),      # 536, in 32 x 32 tiles
    (1, 768, 39, 45, 192, 1, False, False),
    (32, 512, 8, 8, 256, 1, False, True),       # 2 048 pixels
    (33, 512, 8, 8, 256, 1, False, False),
    (4, 512, 36, 37, 64, 2, False, False),      # stride 2, long runs under small tiles
    (3, 512, 38, 38, 128, 1, True, False),      # the pool's second largest tiles
    (2, 512, 38, 38, 128, 1, True, True),
])
def test_where_the_kernel_before_is_ahead(n, ic, h, w, oc, stride, pool, takes, dev, monkeypatch):
    test_tiles_and_lines(n, ic, h, w, oc, stride, pool, takes, dev, monkeypatch)

"""Kernels of the int32 operator contract at the edges of their splits, against the oracle: long reductions, operand packing
of a convolution, depthwise planes."""
import ctypes
import json
import sys
import threading
import time

import numpy as np
import pytest
import torch

import bench
import oracle
from cvm_runtime_amd import check, hipops, lib, synth

pytestmark = pytest.mark.gpu


def T(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("op", ["sum", "max"])
@pytest.mark.parametrize("outputs,run", [(1, 513), (3, 1023), (2, 1024), (5, 1025), (7, 4099), (300, 3136), (1, 70001)])
def test_long_runs(op, outputs, run, dev):
    x = synth.tensor("runs", "%d-%d" % (outputs, run), (outputs, run), -2 ** 31, 2 ** 31 - 1)
    x[0] = -np.abs(x[0] // 2) - 1   # all negative
    got = hipops.reduce(op, T(x, dev), (1,)).cpu().numpy()
    assert np.array_equal(got, oracle.reduce(op, x, (1,)))


@pytest.mark.parametrize("n,c,h,w,oc,k", [(1, 17, 1, 1, 5, 1), (2, 33, 7, 9, 40, 3), (3, 64, 5, 13, 32, 1), (1, 100, 8, 8, 130, 3)])
def test_conv_operand_packing(n, c, h, w, oc, k, dev):
    x = synth.tensor("packing", "x%d" % c, (n, c, h, w), -300, 300)   # narrowed like the reference narrows
    wt = synth.tensor("packing", "w%d" % c, (oc, c, k, k), -127, 127)
    got = hipops.conv2d(T(x, dev), T(wt, dev), None, (1, 1), (k // 2, k // 2)).cpu().numpy()
    assert np.array_equal(got, oracle.conv2d(x, wt, None, (1, 1), (k // 2, k // 2)))


@pytest.mark.parametrize("n,c,h,w,oc,k,strides,padding,dilation", [
    # one launch, K split over a workgroup: halves of the channels of 1 and 0, 1 and 1, 2 and 1; ends of K inside a chunk
    (1, 1, 1, 4, 1, 1, (1, 1), (0, 0), (1, 1)), (1, 2, 3, 5, 33, 1, (1, 1), (0, 0), (1, 1)), (2, 3, 9, 7, 32, 3, (1, 1), (1, 1), (1, 1)),
    (1, 31, 6, 6, 31, 1, (1, 1), (1, 1), (1, 1)), (3, 33, 5, 13, 65, 1, (2, 2), (0, 0), (1, 1)), (1, 640, 8, 4, 34, 1, (1, 1), (0, 0), (1, 1)),
    (1, 71, 11, 9, 40, 3, (1, 2), (2, 1), (2, 1)), (2, 64, 12, 12, 64, 3, (2, 2), (0, 0), (1, 1)), (1, 17, 40, 3, 5, 3, (1, 1), (3, 4), (1, 3)),
    # beyond the tiles of that: filters in LDS, one and two rounds of pixel groups, a last group of few pixels
    (5, 20, 41, 37, 80, 1, (1, 1), (0, 0), (1, 1)), (1, 255, 50, 51, 200, 1, (1, 1), (0, 0), (1, 1)), (16, 33, 57, 57, 130, 1, (1, 1), (0, 0), (1, 1)),
    (4, 256, 33, 32, 129, 1, (2, 1), (1, 0), (1, 1)),
    # the first sizes of the general path: K of 641 and 257, tiles
    (1, 641, 8, 4, 34, 1, (1, 1), (0, 0), (1, 1)), (1, 257, 60, 64, 128, 1, (1, 1), (0, 0), (1, 1)), (2, 64, 56, 57, 64, 3, (1, 1), (1, 1), (1, 1)),
])
def test_conv_direct(n, c, h, w, oc, k, strides, padding, dilation, dev):
    cid = "direct-%d-%d-%d-%d" % (c, h, w, oc)
    x = synth.tensor(cid, "x", (n, c, h, w), -300, 300)   # narrowed like the reference narrows
    wt = synth.tensor(cid, "w", (oc, c, k, k), -300, 300)
    b = synth.tensor(cid, "b", (oc,), -2 ** 31, 2 ** 31 - 1)
    for bias in (None, b):
        got = hipops.conv2d(T(x, dev), T(wt, dev), None if bias is None else T(b, dev), strides, padding, dilation).cpu().numpy()
        assert np.array_equal(got, oracle.conv2d(x, wt, bias, strides, padding, dilation))


@pytest.mark.parametrize("m,k,n", [
    (1, 17, 5), (3, 31, 40),       # a granule that ends inside the channels, one that is all padding
    (33, 64, 32), (70, 100, 7),
    (5, 1023, 33),                 # rows that do not start on 16 bytes
    (1, 16416, 4100),              # a filter of so many dwords that the workgroups that pack it go round
])
def test_dense_operand_packing(m, k, n, dev):
    x = synth.tensor("rows", "x%d" % k, (m, k), -127, 127)
    wt = synth.tensor("rows", "w%d" % k, (n, k), -127, 127)
    got = hipops.dense(T(x, dev), T(wt, dev)).cpu().numpy()
    assert np.array_equal(got, oracle.dense(x, wt, None))
    packed = hipops.unpack_act_i8(hipops.pack_act_i8(T(x.reshape(m, k, 1, 1), dev)), m, k, 1, 1).cpu().numpy()
    assert np.array_equal(packed.reshape(m, k), x)


@pytest.mark.parametrize("n,c,h,w,oc,k,kernels", [
    (1, 256, 14, 15, 65, 1, {"k_conv_direct"}),
    (1, 64, 14, 15, 65, 3, {"k_conv_direct"}),
    (4, 96, 61, 75, 160, 1, {"k_conv_slab"}),
    (1, 128, 28, 28, 64, 3, {"k_pack_both", "k_conv_wave"}),
    (1, 16, 28, 28, 64, 5, {"k_pack_act", "k_conv_igemm"}),   # few channels
])
def test_every_form_of_conv2d_is_timed(n, c, h, w, oc, k, kernels, dev):
    """The launches between cvmhip_kernel_timing_begin and _end, with the work and the bytes of the layer."""
    x, wt = T(synth.tensor("timed", "x%d" % c, (n, c, h, w), -127, 127), dev), T(synth.tensor("timed", "w%d" % c, (oc, c, k, k), -127, 127), dev)
    ends = {}
    for name in ("cvmhip_kernel_timing_end", "cvmhip_kernel_timing_end_launches"):
        check(lib().cvmhip_kernel_timing_begin())
        for _ in range(3):
            y = hipops.conv2d(x, wt, None, (1, 1), (k // 2, k // 2))
        buf = ctypes.create_string_buffer(1 << 16)
        check(getattr(lib(), name)(buf, len(buf)))
        ends[name] = json.loads(buf.value.decode())
    kt, launches = ends.values()
    assert set(kt) == kernels == {e["kernel"] for e in launches}
    dominant = bench.dominant_conv(kt, 0.0, 3)
    assert dominant["kernel"] in kernels and dominant["kernel"].startswith("k_conv")
    assert dominant["conv"]["launches"] == 3 and dominant["conv"]["ms"] > 0 and dominant["ops_per_launch"] == pytest.approx(2 * y.numel() * c * k * k, rel=1e-5)
    one = [e for e in launches if e["kernel"] == dominant["kernel"]][0]
    assert "%dx%d/1 %d->%d in %dx%dx%d out %dx%d" % (k, k, c, oc, n, h, w, h, w) in one["desc"] and one["ms"] > 0
    if len(kernels) == 1:
        assert one["bytes"] == pytest.approx(4 * (x.numel() + wt.numel() + y.numel()), rel=1e-5)   # (written with seven digits)


@pytest.mark.parametrize("n,c,mult,h,w,strides,padding,dilation", [
    (1, 2, 1, 3, 3, (1, 1), (0, 0), (1, 1)),       # one output
    (2, 3, 2, 5, 7, (1, 1), (1, 1), (1, 1)),       # a channel multiplier; rows that are not whole quads
    (1, 5, 1, 9, 6, (2, 2), (1, 1), (1, 1)),
    (1, 4, 1, 12, 11, (1, 2), (2, 3), (2, 1)),
    (1, 4, 1, 12, 70, (2, 1), (0, 2), (1, 3)),
    (3, 130, 1, 33, 64, (1, 1), (1, 1), (1, 1)),   # several workgroups per plane
])
def test_depthwise_planes(n, c, mult, h, w, strides, padding, dilation, dev):
    x = synth.tensor("planes", "x%d-%d" % (c, w), (n, c, h, w), -2 ** 31, 2 ** 31 - 1)   # exact and wrapping
    wt = synth.tensor("planes", "w%d-%d" % (c, w), (c * mult, 1, 3, 3), -2 ** 31, 2 ** 31 - 1)
    b = synth.tensor("planes", "b%d" % c, (c * mult,), -32768, 32768)
    got = hipops.conv2d(T(x, dev), T(wt, dev), T(b, dev), strides, padding, dilation, groups=c).cpu().numpy()
    assert np.array_equal(got, oracle.conv2d(x, wt, b, strides, padding, dilation, groups=c))


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("n,c,h,w", [(1, 1, 1, 1), (1, 3, 2, 5), (2, 5, 7, 6), (1, 70, 19, 75), (4, 70, 64, 61)])   # the last: four rows a thread
@pytest.mark.parametrize("last", [0, 2 ** 23])   # all values in 24 bits; one that is not, in the last wavefront
def test_depthwise_planes_narrow(n, c, h, w, stride, last, dev):
    x = synth.tensor("narrow", "x%d-%d" % (c, w), (n, c, h, w), -2 ** 23, 2 ** 23 - 1)
    wt = synth.tensor("narrow", "w%d" % c, (c, 1, 3, 3), -2 ** 23, 2 ** 23 - 1)
    if last:
        x[-1, -1, -1, -1] = last
    wt[0, 0, 1, 1], x[0, 0, 0, 0] = -2 ** 23, 2 ** 23 - 1
    got = hipops.conv2d(T(x, dev), T(wt, dev), None, (stride, stride), (1, 1), groups=c).cpu().numpy()
    assert np.array_equal(got, oracle.conv2d(x, wt, None, (stride, stride), (1, 1), (1, 1), groups=c))


@pytest.mark.parametrize("widths,outer,inner", [
    ((1, 1, 4), 24564, 1),                          # a detector's rows
    ((3,), 5, 7),
    ((1,) * 8, 3, 1), ((2,) * 9, 257, 3),           # a whole group, one more
    ((5, 0, 1, 300, 2), 11, 2),
])
def test_concat_groups(widths, outer, inner, dev):
    xs = [synth.tensor("concat", "x%d-%d" % (i, w), (outer, max(w, 1), inner), -2 ** 31, 2 ** 31 - 1)[:, :w] for i, w in enumerate(widths)]
    got = hipops.concatenate([T(x, dev) for x in xs], 1).cpu().numpy()
    assert np.array_equal(got, np.concatenate(xs, 1))


def test_other_threads_run_during_an_operator_call(dev):
    """The interpreter's lock is free while the library issues a launch: with switching by time all but off, another
    thread gets on only if the calls let it."""
    x = T(np.arange(64, dtype=np.int32), dev)
    y = hipops.relu(x)   # written again by every call: an allocation or a release of its own could let go of the lock
    seen, started, stop = [0], threading.Event(), threading.Event()

    def other():
        started.set()
        while not stop.is_set():
            seen[0] += 1
            time.sleep(0)
    t = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    t.start()
    started.wait()
    sys.setswitchinterval(1000.0)
    try:
        before = seen[0]
        for _ in range(5000):
            hipops.relu(x, y)
            if seen[0] >= before + 20:   # (a wait that began before the interval was set ends once more)
                break
        moved = seen[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        t.join()
    assert moved >= 20


@pytest.mark.parametrize("n,c,h,w,oc,stride,padding", [
    (1, 33, 130, 128, 1, (1, 1), (0, 0)),      # one channel of a tile of 32; chunks that end inside a half of the channels
    (3, 16, 90, 91, 31, (1, 1), (0, 0)),       # one chunk; several rounds of pixels to a workgroup
    (1, 255, 61, 60, 128, (1, 1), (0, 0)),     # 64 would be few workgroups; eight chunks, the last one short
    (2, 160, 75, 75, 96, (1, 1), (1, 1)),      # the last 64 channels half past the end; five chunks, a border
    (9, 96, 57, 63, 150, (1, 1), (0, 0)),      # beyond, both in rounds
    (10, 64, 75, 75, 224, (1, 1), (0, 0)),     # 64 channels to a workgroup: two chunks, half of the four in flight
    (8, 200, 70, 61, 192, (1, 1), (0, 1)),     # seven chunks
    (8, 100, 95, 96, 256, (2, 2), (0, 0)),     # stride 2
])
def test_conv_slab_widths(n, c, h, w, oc, stride, padding, dev):
    cid = "slab-%d-%d-%d-%d" % (c, h, w, oc)
    x = synth.tensor(cid, "x", (n, c, h, w), -300, 300)   # narrowed like the reference narrows
    wt = synth.tensor(cid, "w", (oc, c, 1, 1), -300, 300)
    b = synth.tensor(cid, "b", (oc,), -2 ** 31, 2 ** 31 - 1)
    for bias in (None, b):
        got = hipops.conv2d(T(x, dev), T(wt, dev), None if bias is None else T(b, dev), stride, padding).cpu().numpy()
        assert np.array_equal(got, oracle.conv2d(x, wt, bias, stride, padding))


@pytest.mark.parametrize("n,c,h,w,oc,padding", [
    (6, 24, 75, 75, 64, (0, 0)),        # 64 channels and two chunks in flight: one chunk a group, one round
    (10, 112, 86, 80, 64, (0, 0)),      # four chunks, two rounds
    (6, 100, 74, 75, 60, (1, 0)),       # with a border
    (10, 48, 86, 80, 32, (0, 0)),       # 32 channels and two in flight, in rounds
    (5, 48, 70, 70, 200, (0, 0)),       # 32 and four, a round more than with 64
    (12, 50, 96, 96, 64, (0, 0)),       # 64 and four, one workgroup to its pixels
    (2, 256, 60, 60, 96, (1, 1)),       # 32 and four, with a border
])
def test_conv_slab_chunks_in_flight(n, c, h, w, oc, padding, dev):
    cid = "slab-%d-%d-%d-%d" % (c, h, w, oc)
    x = synth.tensor(cid, "x", (n, c, h, w), -300, 300)
    wt = synth.tensor(cid, "w", (oc, c, 1, 1), -300, 300)
    b = synth.tensor(cid, "b", (oc,), -2 ** 31, 2 ** 31 - 1)
    got = hipops.conv2d(T(x, dev), T(wt, dev), T(b, dev), (1, 1), padding).cpu().numpy()
    assert np.array_equal(got, oracle.conv2d(x, wt, b, (1, 1), padding))

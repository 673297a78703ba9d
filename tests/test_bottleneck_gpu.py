"""The 3x3 layer of a bottleneck, the 1x1 layer behind it with the residual and the next block's first layer in one launch, against the oracle
running the graph node by node."""
import ctypes
import json

import numpy as np
import pytest

import oracle
import oracle.graph as og
from cvm_runtime_amd import check, graphgen, hipops, lib, runtime, synth
from cvm_runtime_amd.hipops import chain


class Projection(ctypes.Structure):
    _fields_ = [("x", ctypes.c_void_p), ("w", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("chain", ctypes.POINTER(hipops.Chain)), ("c", ctypes.c_int)]


def _clamp_shift(lo, hi, shift):
    c = hipops.Chain()
    c.count = 1
    c.stage[0] = hipops.Stage(5, 0, shift, lo, hi)
    return c


def _net(n, m, h, w, oc, stride, multiply=False, reader=False, projects=False):
    g = graphgen.GraphBuilder("bottleneck-%d-%d-%d" % (m, oc, stride))
    x0 = g.conv_relu_q(g.var("data", (n, 32, h, w), 8), 64 if m == 64 else 2 * m, 1)
    x = g.conv_relu_q(x0, m, 1)
    if not projects:   # another reader of the residual keeps its 1x1 layer apart
        r = g.conv_relu_q(x0, 4 * m, 1, stride, 0, relu=False)
    y, k = g.conv(x, m, 3, stride, 1)
    if multiply:   # a chain that is no clamp and shift
        y = g.op("broadcast_mul", [y, g.param("m", (1,), 3, 3, 3)], {}, [g.shape(y)])[0]
    y = a = g.rshift(g.relu(y), graphgen.shift_for(k) + 2 * multiply)
    z = g.conv_relu_q(y, 4 * m, 1, relu=False)
    if projects:
        r = g.conv_relu_q(x0, 4 * m, 1, stride, 0, relu=False)
    y = g.rshift(g.relu(g.add(z, r)), 1)
    z = g.conv_relu_q(y, oc, 1)
    # everything the launch stores is read again, as int8
    tails = [g.conv_relu_q(z, 16, 1, relu=False), g.conv_relu_q(y, 16, 1, relu=False)] + ([g.conv_relu_q(a, 16, 1, relu=False)] if reader else [])
    if not projects:
        tails.append(g.conv_relu_q(r, 16, 1, relu=False))
    out = tails[0]
    for t in tails[1:]:
        out = g.concat([out, t], 1)
    return g.build([out])


def _run(js, pb, data, monkeypatch, calls=3):
    """outputs of some calls (eager, captured, replayed), and the launches of a run with and without the launch in question"""
    monkeypatch.setenv("CVM_HIP_RESIDENT", "1")   # no layer sequences: a measurement at load would choose
    m = runtime.HipModel(js, pb)
    launches = [m.launch_counts()[0]]
    got = [np.frombuffer(m.inference(data.astype(np.int8).tobytes()), np.int8) for _ in range(calls)]
    m.close()
    monkeypatch.setenv("CVM_HIP_SEPARABLE", "0")
    m = runtime.HipModel(js, pb)
    launches.append(m.launch_counts()[0])
    m.close()
    return got, launches


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,h,w,oc,stride", [
    (1, 64, 1, 1, 64, 1),            # one pixel: every window leaves the image on all sides
    (1, 64, 2, 3, 128, 2),
    (2, 64, 13, 9, 64, 1),           # tiles that span images and end in the last one
    (5, 64, 56, 56, 128, 1),         # tiles of 64 pixels, the last one whole
    (2, 64, 127, 97, 64, 1),         # of 128
    (3, 64, 101, 113, 128, 1),       # of 128
    (9, 64, 113, 111, 64, 2),
    (1, 128, 7, 5, 256, 1),          # of 16
    (2, 128, 56, 56, 128, 2),
    (3, 128, 41, 37, 128, 1),        # of 32
    (7, 128, 37, 37, 256, 1),        # of 48
    (17, 128, 28, 28, 128, 1),       # of 64, one to a compute unit
    (23, 128, 28, 29, 128, 1),       # of 80
    (29, 128, 29, 28, 256, 1),       # of 96
    (33, 128, 28, 28, 128, 1),       # of 64 again
    (20, 128, 60, 56, 128, 2),       # stride 2: of 80
    (1, 256, 3, 14, 256, 1),         # of 16
    (5, 256, 28, 28, 512, 2),
    (22, 256, 14, 15, 256, 1),       # of 32
    (45, 256, 14, 14, 512, 1),       # of 48
    (43, 256, 28, 28, 256, 2),       # of 48, the longest run of the input
    (64, 256, 14, 14, 256, 1),       # of 64
])
def test_bottleneck_in_one_launch(n, m, h, w, oc, stride, dev):
    import torch
    bias = n > 1   # with one image: none
    rng = np.random.default_rng(n * h * w + m)
    oh, ow = (h - 1) // stride + 1, (w - 1) // stride + 1
    shapes = {"a": (m, m, 3, 3), "b": (4 * m, m, 1, 1), "c": (oc, 4 * m, 1, 1)}
    x, r = (rng.integers(-128, 128, v, dtype=np.int32) for v in ((n, m, h, w), (n, 4 * m, oh, ow)))
    f = {k: rng.integers(-128, 128, v, dtype=np.int32) for k, v in shapes.items()}
    b = {k: rng.integers(-40000, 40000, v[0], dtype=np.int32) if bias else None for k, v in shapes.items()}
    # clamps that act, on both sides, in front of and behind the residual
    sh = {k: graphgen.shift_for(v[1] * v[2] * v[3]) for k, v in shapes.items()}
    q = {"a": (0, (128 << sh["a"]) - 1, sh["a"]), "b": (-300 << sh["b"], (150 << sh["b"]) + 5, sh["b"]), "r": (-200, 255, 1),
         "c": (-(128 << sh["c"]), (127 << sh["c"]) + 3, sh["c"])}

    def requant(v, k):
        return np.clip(v, q[k][0], q[k][1]) >> q[k][2]

    ya = requant(oracle.conv2d(x, f["a"], b["a"], (stride, stride), (1, 1)), "a")
    yb = requant(requant(oracle.conv2d(ya, f["b"], b["b"]), "b") + r, "r")
    yc = requant(oracle.conv2d(yb, f["c"], b["c"]), "c")

    def dt(v):
        return torch.from_numpy(np.ascontiguousarray(v)).to(dev)

    xp, rp = hipops.pack_act_i8(dt(x)), hipops.pack_act_i8(dt(r))
    wp = {k: hipops.pack_weights(dt(v)) for k, v in f.items()}
    bp = {k: dt(v) if bias else None for k, v in b.items()}
    out, nxt = hipops._act_buffer(n * oh * ow, 4 * m, dev), hipops._act_buffer(n * oh * ow, oc, dev)
    c = {k: _clamp_shift(*v) for k, v in q.items()}
    vp, ref = hipops._vp, ctypes.byref
    # a later launch's filters, of which nothing but their bytes is used (there is no later one)
    class Filters(ctypes.Structure):
        _fields_ = [(k, ctypes.c_void_p) for k in ("wa", "wb", "wc")] + [("m", ctypes.c_int), ("oc", ctypes.c_int)]
    ahead = ref(Filters(wp["a"].data_ptr(), wp["b"].data_ptr(), wp["c"].data_ptr(), m, oc)) if n % 2 else None
    check(lib().cvmhip_conv2d_bottleneck_i8(vp(xp), vp(wp["a"]), vp(bp["a"]), ref(c["a"]), vp(wp["b"]), vp(bp["b"]), ref(c["b"]), vp(rp), ref(c["r"]),
                                            vp(out), vp(wp["c"]), vp(bp["c"]), ref(c["c"]), vp(nxt), n, m, h, w, oc, stride, None, ahead, hipops._conv_stream()))
    assert np.array_equal(hipops.unpack_act_i8(out, n, 4 * m, oh, ow).cpu().numpy(), yb)
    assert np.array_equal(hipops.unpack_act_i8(nxt, n, oc, oh, ow).cpu().numpy(), yc)
    if oc != m or not _eligible(n, m, h, w, oc, stride, _projection(64 if m == 64 else 2 * m)):
        return
    # the residual made by a projection of the block's input
    cs = 64 if m == 64 else 2 * m
    f["s"] = rng.integers(-128, 128, (4 * m, cs, 1, 1), dtype=np.int32)
    b["s"] = rng.integers(-40000, 40000, 4 * m, dtype=np.int32) if bias else None
    sh = graphgen.shift_for(cs)
    q["s"] = (-(128 << sh), (127 << sh) + 3, sh)
    xs = rng.integers(-128, 128, (n, cs, h, w), dtype=np.int32)
    yb = requant(requant(oracle.conv2d(ya, f["b"], b["b"]), "b") + requant(oracle.conv2d(xs, f["s"], b["s"], (stride, stride)), "s"), "r")
    yc = requant(oracle.conv2d(yb, f["c"], b["c"]), "c")
    xsp, ws, bs, chain_s = hipops.pack_act_i8(dt(xs)), hipops.pack_weights(dt(f["s"])), dt(b["s"]) if bias else None, _clamp_shift(*q["s"])

    projection = Projection(xsp.data_ptr(), ws.data_ptr(), bs.data_ptr() if bias else None, ctypes.pointer(chain_s), cs)
    out.zero_()
    nxt.zero_()
    check(lib().cvmhip_conv2d_bottleneck_i8(vp(xp), vp(wp["a"]), vp(bp["a"]), ref(c["a"]), vp(wp["b"]), vp(bp["b"]), ref(c["b"]), None, ref(c["r"]),
                                            vp(out), vp(wp["c"]), vp(bp["c"]), ref(c["c"]), vp(nxt), n, m, h, w, oc, stride, ref(projection), ahead,
                                            hipops._conv_stream()))
    assert np.array_equal(hipops.unpack_act_i8(out, n, 4 * m, oh, ow).cpu().numpy(), yb)
    assert np.array_equal(hipops.unpack_act_i8(nxt, n, oc, oh, ow).cpu().numpy(), yc)


@pytest.mark.gpu
@pytest.mark.parametrize("projects", [False, True])
@pytest.mark.parametrize("n,m,h,w,oc,stride", [(2, 64, 40, 41, 64, 1), (1, 128, 57, 56, 128, 2), (1, 128, 57, 56, 256, 2), (3, 256, 28, 26, 256, 1)])
def test_bottleneck_of_a_graph(n, m, h, w, oc, stride, projects, dev, monkeypatch):
    js, pb = _net(n, m, h, w, oc, stride, projects=projects)
    data = synth.tensor("bottleneck", "data%d" % (h * w), (n, 32, h, w), -128, 127)
    got, launches = _run(js, pb, data, monkeypatch)
    # of the layers apart, some may share a launch with one that does not depend on them
    assert launches[0] < launches[1] and (not projects or oc != m or launches[0] <= launches[1] - 2), launches
    want = og.run_graph(js, graphgen.load_params(pb), data.astype(np.int32))[0].ravel()
    assert all(np.array_equal(v.astype(np.int32), want) for v in got)


@pytest.mark.gpu
@pytest.mark.parametrize("multiply,reader", [(True, False), (False, True)])
def test_layers_that_stay_apart(multiply, reader, dev, monkeypatch):
    """A chain with a multiplication, and a 3x3 result that another layer reads."""
    js, pb = _net(2, 64, 20, 20, 64, 1, multiply, reader)
    data = synth.tensor("bottleneck", "apart", (2, 32, 20, 20), -128, 127)
    got, launches = _run(js, pb, data, monkeypatch)
    assert launches[1] == launches[0], launches
    want = og.run_graph(js, graphgen.load_params(pb), data.astype(np.int32))[0].ravel()
    assert all(np.array_equal(v.astype(np.int32), want) for v in got)


def _projection(c, chain_s=None):
    return ctypes.byref(Projection(None, None, None, ctypes.pointer(chain_s or _clamp_shift(-128 << 5, 127 << 5, 5)), c))


def _eligible(n=1, m=64, h=14, w=14, oc=64, stride=1, projection=None, **chains):
    plain = _clamp_shift(-127 << 9, 127 << 9, 9)
    c = [chains.get(k, plain) for k in ("a", "b", "r", "c")]
    return lib().cvmhip_bottleneck_eligible(n, m, h, w, oc, stride, *[ctypes.byref(v) for v in c], projection)


def test_which_layers_are_taken():
    assert _eligible() and _eligible(m=256, oc=512, stride=2, h=28, w=28, n=50) and _eligible(h=1, w=1)
    for bad in (dict(m=32, oc=32), dict(m=512, oc=512), dict(m=96, oc=96), dict(oc=32), dict(oc=192), dict(stride=3), dict(h=0), dict(n=0),
                dict(n=1 << 20, h=64, w=64)):
        assert not _eligible(**bad), bad
    wide = _clamp_shift(-128 << 9, (128 << 9) + 511, 9)   # 128 is no int8
    assert not _eligible(a=wide) and not _eligible(r=wide) and not _eligible(c=wide)
    assert _eligible(b=wide)                      # in front of the residual the sum is 32 bits wide
    for two in (chain(("mul", 3)), chain(("cvm_right_shift", 8, 9)), chain(("mul", 3), ("cvm_right_shift", 8, 9))):
        assert not any(_eligible(**{k: two}) for k in "abrc")
    # a projection of the block's input
    assert _eligible(projection=_projection(64)) and _eligible(m=128, oc=128, projection=_projection(256)) and _eligible(m=256, oc=256, stride=2, projection=_projection(512))
    for bad in (dict(projection=_projection(128)), dict(oc=128, projection=_projection(64)), dict(m=128, oc=128, projection=_projection(64)), dict(projection=_projection(64, wide))):
        assert not _eligible(**bad), bad
    # ... which needs room beside the longest runs of the input
    assert _eligible(n=50, m=256, oc=256, h=28, w=28, stride=2) and not _eligible(n=50, m=256, oc=256, h=28, w=28, stride=2, projection=_projection(512))
    # rows so long that not even the smallest tile's run of the input fits in LDS
    assert _eligible(m=256, oc=256, w=100) and not _eligible(m=256, oc=256, w=400)
    assert not _eligible(m=64, oc=64, w=4000) and not _eligible(m=256, oc=256, w=200, h=200, stride=2)


@pytest.mark.parametrize("m,w", [(128, 1 << 28), (256, 1 << 27), (256, (1 << 27) + 5)])
def test_rows_whose_bytes_do_not_fit_in_32_bits(m, w):
    """The run of the input under the smallest tile is two rows and more: 2 * w * m bytes of LDS, next to nothing in 32 bits."""
    assert 2 * w * m // 16 % 2**32 < 4096
    assert not _eligible(m=m, oc=m, h=1, w=w)


def test_products_of_sizes_past_64_bits():
    """No tensor has such sizes; in 64 bits the pixels are 0 and the bytes 2^30."""
    assert (1 << 30) * (1 << 30) * 16 % 2**64 == 0 and 652805 * 26317 * (1 << 30) % 2**64 == 1 << 30
    assert not _eligible(n=1 << 30, h=1 << 30, w=16) and not _eligible(n=1 << 30, h=1 << 30, w=16, stride=2)
    c, size = _clamp_shift(0, 127 << 12, 12), dict(n=652805, ic=1 << 30, h=26317, w=1)
    run = [lib().cvmhip_conv2d_run_eligible(ctypes.byref(c), v["n"], v["ic"], v["h"], v["w"], 64, 3, 3, 1, 1, 1, 1, 1, 1) for v in (size, dict(size, n=1, h=7, ic=512))]
    assert not run[0] and run[1]


def test_longest_run_of_a_stride_2_layer():
    """Against the runs of all tiles: whether the smallest tile's fits in LDS with the results and the biases."""
    rng, taken = np.random.default_rng(7), 0
    for _ in range(400):
        m, n, h, w = int(rng.choice([64, 128, 256])), int(rng.integers(1, 6)), int(rng.integers(1, 40)), int(rng.integers(1, 90) * rng.integers(1, 12))
        pixels, oh, ow = 32 if m == 64 else 16, (h + 1) // 2, (w + 1) // 2
        p = np.arange(0, n * oh * ow, pixels)
        first, last = (((q // (oh * ow)) * h + q % (oh * ow) // ow * 2 - 1) * w + q % ow * 2 - 1 for q in (p, np.minimum(p + pixels, n * oh * ow) - 1))
        run = int((last + 2 * w + 2 - first + 1).max())
        lds = 64 + -(-6 * m * 4 // 1024) * 1024 + 5 * m // 16 * pixels * 16 + -(-run * (m // 16) // 64) * 1024
        assert bool(_eligible(n=n, m=m, oc=m, h=h, w=w, stride=2)) == (lds <= 160 * 1024), (n, m, h, w)
        taken += lds <= 160 * 1024
    assert 100 < taken < 390


def _launches(run):
    """What the launches of `run` say of themselves"""
    L = lib()
    L.cvmhip_kernel_timing_begin()
    run()
    check(L.cvmhip_device_sync())
    buf = ctypes.create_string_buffer(1 << 18)
    check(L.cvmhip_kernel_timing_end_launches(buf, len(buf)))
    return [str(v) for v in json.loads(buf.value.decode())]


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,h,w,oc,tile,projected", [
    (2, 64, 13, 9, 64, 32, 32), (2, 64, 13, 9, 128, 32, None),
    (3, 64, 57, 61, 64, 64, 64), (3, 64, 57, 61, 128, 64, None),
    (2, 64, 101, 99, 64, 96, 96), (2, 64, 101, 99, 128, 96, None),
    (3, 64, 93, 91, 64, 128, 128), (3, 64, 93, 91, 128, 128, None),
    (1, 128, 7, 5, 128, 16, 16), (1, 128, 7, 5, 256, 16, None),
    (3, 128, 41, 37, 128, 32, 32), (3, 128, 41, 37, 256, 32, None),
    (7, 128, 37, 37, 128, 48, 48), (7, 128, 37, 37, 256, 48, None),
    (17, 128, 28, 28, 128, 64, 64), (17, 128, 28, 28, 256, 64, None),
    (23, 128, 28, 29, 128, 80, 80), (23, 128, 28, 29, 256, 80, None),
    (29, 128, 29, 28, 128, 96, 96), (29, 128, 29, 28, 256, 96, None),
    (32, 128, 28, 28, 128, 64, 64), (32, 128, 28, 28, 256, 64, None),
    (1, 256, 3, 14, 256, 16, 16), (1, 256, 3, 14, 512, 16, None),
    (22, 256, 14, 15, 256, 32, 32), (22, 256, 14, 15, 512, 32, None),
    (45, 256, 14, 14, 256, 48, 48), (45, 256, 14, 14, 512, 48, None),
    (63, 256, 14, 14, 256, 64, 64), (63, 256, 14, 14, 512, 64, None),
])
def test_every_form(n, m, h, w, oc, tile, projected, dev):
    """Each tile with each third layer, and with the projection (or without, where that leaves a smaller tile only)."""
    said = [v for v in _launches(lambda: test_bottleneck_in_one_launch(n, m, h, w, oc, 1, dev)) if "k_conv_block" in v]
    assert "tile %d " % tile in said[0] and "+res" in said[0], said
    assert len(said) == 1 + (projected is not None), said
    if projected:
        assert "tile %d " % projected in said[1] and "+ projection" in said[1], said


@pytest.mark.gpu
@pytest.mark.parametrize("m,oc,projects", [(128, 128, False), (128, 256, False), (128, 128, True), (256, 256, False), (256, 512, False), (256, 256, True)])
@pytest.mark.parametrize("later_oc", [256, 512])
def test_filters_of_the_next_launch(m, oc, projects, later_oc, dev):
    """Idle compute units read the next launch's filters: the results are what they are without."""
    import torch
    n, h, w, gen = 2, 15, 13, torch.Generator(device=dev)
    gen.manual_seed(m + oc)
    c = 2 * m
    rand = lambda *s: torch.randint(-128, 128, s, dtype=torch.int32, device=dev, generator=gen)
    x, r, xs = hipops.pack_act_i8(rand(n, m, h, w)), hipops.pack_act_i8(rand(n, 4 * m, h, w)), hipops.pack_act_i8(rand(n, c, h, w))
    wa, wb, wc, ws = (hipops.pack_weights(rand(*s)) for s in ((m, m, 3, 3), (4 * m, m, 1, 1), (oc, 4 * m, 1, 1), (4 * m, c, 1, 1)))
    la, lb, lc = (hipops.pack_weights(rand(*s)) for s in ((256, 256, 3, 3), (1024, 256, 1, 1), (later_oc, 1024, 1, 1)))

    class Filters(ctypes.Structure):
        _fields_ = [(k, ctypes.c_void_p) for k in ("wa", "wb", "wc")] + [("m", ctypes.c_int), ("oc", ctypes.c_int)]
    chains = [_clamp_shift(-(127 << s), 127 << s, s) for s in (12, 10, 1, 12, 10)]
    ca, cb, cr, cc = (ctypes.byref(v) for v in chains[:4])
    projection = ctypes.byref(Projection(xs.data_ptr(), ws.data_ptr(), None, ctypes.pointer(chains[4]), c)) if projects else None
    outs = []
    for ahead in (None, Filters(la.data_ptr(), lb.data_ptr(), lc.data_ptr(), 256, later_oc), Filters(None, lb.data_ptr(), None, 256, later_oc)):
        out, nxt = hipops._act_buffer(n * h * w, 4 * m, dev), hipops._act_buffer(n * h * w, oc, dev)
        vp = hipops._vp
        said = _launches(lambda: check(lib().cvmhip_conv2d_bottleneck_i8(
            vp(x), vp(wa), None, ca, vp(wb), None, cb, None if projects else vp(r), cr, vp(out), vp(wc), None, cc, vp(nxt), n, m, h, w, oc, 1,
            projection, ctypes.byref(ahead) if ahead else None, hipops._conv_stream())))
        assert "+ %d ahead" % (64 if ahead else 0) in said[-1], said
        outs.append((hipops.unpack_act_i8(out, n, 4 * m, h, w), hipops.unpack_act_i8(nxt, n, oc, h, w)))
    for a, b in outs[1:]:
        assert torch.equal(a, outs[0][0]) and torch.equal(b, outs[0][1])


@pytest.mark.gpu
def test_several_blocks_of_a_graph(dev, monkeypatch):
    """Blocks one behind the other, through a change of their width: where compute units are idle a launch has the next one's filters fetched."""
    g, heads = graphgen.resnet50(13, blocks=(1, 2, 3, 1), size=96, classes=40, config_id="bottlenecks")   # 468 pixels of 256 channels
    js, pb = g.build(heads)
    monkeypatch.setenv("CVM_HIP_RESIDENT", "1")
    m = runtime.HipModel(js, pb)
    inputs = [synth.tensor("bottlenecks", "data%d" % k, (13, 3, 96, 96), -127, 127) for k in range(2)]
    wants = [og.run_graph(js, graphgen.load_params(pb), x)[0].ravel() for x in inputs]
    for call in range(4):
        assert np.array_equal(np.frombuffer(m.inference(inputs[call % 2].astype(np.int8).tobytes()), np.int32), wants[call % 2]), call
    said = [v for v in _launches(m.run) if "k_conv_block" in v]
    assert len(said) == 6 and sum("+ 64 ahead" in v for v in said) == 2, said
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("spin", ["", "0"])   # "0": every wait of the sequence gives up, and the run is repeated without it
def test_beside_a_sequence(spin, dev, monkeypatch):
    """The block's projection is too large for a layer sequence, which begins behind it: with sequences the projection is a launch of its own, without
    them (another such model is loaded, or the sequence gave up) all four layers are one."""
    js, pb = _net(66, 256, 14, 14, 256, 1, projects=True)
    inputs = [synth.tensor("bottleneck", "seq%d" % k, (66, 32, 14, 14), -128, 127).astype(np.int8) for k in range(3)]
    monkeypatch.setenv("CVM_HIP_SEPARABLE", "0")
    monkeypatch.setenv("CVM_HIP_SEQ", "0")
    m = runtime.HipModel(js, pb)
    wants = [m.inference(x.tobytes()) for x in inputs]
    m.close()
    monkeypatch.setenv("CVM_HIP_SEQ", "1")
    monkeypatch.setenv("CVM_HIP_SEPARABLE", "1")
    if spin:
        monkeypatch.setenv("CVM_HIP_SEQ_SPIN", spin)
    m = runtime.HipModel(js, pb)
    counts = [m.launch_counts()]
    assert counts[0][1] == 1 and counts[0][2] >= 3
    for k in range(4):
        assert m.inference(inputs[k % 3].tobytes()) == wants[k % 3], k
    if spin:
        assert m.launch_counts()[1] == 0
    else:
        assert not any("k_conv_block" in v for v in _launches(m.run))
        other = runtime.HipModel(js, pb)
        for k in range(4):
            assert m.inference(inputs[k % 3].tobytes()) == wants[k % 3], k
        assert any("+ projection" in v for v in _launches(m.run))
        other.close()
        for k in range(4):
            assert m.inference(inputs[k % 3].tobytes()) == wants[k % 3], k
    m.close()


@pytest.mark.gpu
def test_few_pixels_stay_apart(dev, monkeypatch):
    js, pb = _net(2, 256, 14, 14, 256, 1, projects=True)
    data = synth.tensor("bottleneck", "few", (2, 32, 14, 14), -128, 127)
    got, launches = _run(js, pb, data, monkeypatch)
    assert launches[0] == launches[1], launches
    want = og.run_graph(js, graphgen.load_params(pb), data.astype(np.int32))[0].ravel()
    assert all(np.array_equal(v.astype(np.int32), want) for v in got)


def test_which_launches_gain():
    def gains(n, m, h, w, oc, stride, projection=None):
        assert _eligible(n, m, h, w, oc, stride, projection)
        return bool(lib().cvmhip_bottleneck_gains(n, m, h, w, oc, stride, projection))
    for n, m, h, w, oc, stride in ((3, 256, 14, 14, 256, 1), (50, 256, 28, 28, 512, 2), (1, 256, 59, 59, 256, 1), (1, 128, 7, 7, 128, 1), (1, 64, 1, 1, 64, 1), (256, 64, 56, 56, 128, 1),
                                   (256, 128, 56, 56, 128, 2), (1, 128, 266, 266, 256, 2), (1, 128, 319, 319, 128, 1), (1, 64, 654, 654, 64, 2)):
        assert gains(n, m, h, w, oc, stride), (n, m, h, w)
    for n, m, h, w, oc, stride in ((1, 256, 14, 14, 256, 1), (2, 256, 28, 28, 512, 2), (1, 256, 224, 224, 512, 2), (1, 256, 235, 235, 256, 1), (1, 64, 702, 702, 64, 2), (1, 128, 340, 340, 256, 2),
                                   (1, 128, 328, 516, 128, 1), (1, 128, 331, 331, 128, 1)):
        assert not gains(n, m, h, w, oc, stride), (n, m, h, w)
    assert gains(3, 256, 28, 28, 256, 2, _projection(512)) and not gains(1, 256, 14, 14, 256, 1, _projection(512))
    assert not lib().cvmhip_bottleneck_gains(1, 256, 1, 400, 256, 1, None)   # fits nowhere

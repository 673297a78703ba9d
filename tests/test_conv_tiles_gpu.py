"""Large-tile convolution kernel with the 128 x 128 tile, which the dispatch takes for layers of too few pixels for the
128 x 256 one: edges of the tile, against the oracle, and the lines of the dispatch."""
import ctypes
import json

import numpy as np
import pytest
import torch

import oracle
from cvm_runtime_amd import check, hipops, lib, synth

pytestmark = pytest.mark.gpu


def T(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(dev)


@pytest.fixture
def tile(monkeypatch):
    monkeypatch.setenv("CVM_HIP_CONV", "big")
    monkeypatch.setenv("CVM_HIP_TILE", "4,0")


@pytest.mark.parametrize("n,ic,h,w,oc,k,stride,residual", [
    (9, 64, 32, 32, 256, 3, 1, False),     # whole tiles
    (11, 512, 29, 29, 200, 1, 1, True),    # pixels and channels that end inside a tile, shortest K, residual
    (47, 96, 28, 28, 130, 3, 2, False),    # two channels in the last tile, K of 864
])
def test_tile_128_by_128(n, ic, h, w, oc, k, stride, residual, dev, tile):
    cid = "tile128-%d-%d" % (n, ic)
    x = synth.tensor(cid, "x", (n, ic, h, w), -127, 127)
    wt = synth.tensor(cid, "w", (oc, ic, k, k), -127, 127)
    b = synth.tensor(cid, "b", (oc,), -32768, 32768)
    ref = oracle.cvm_right_shift(oracle.relu(oracle.conv2d(x, wt, b, (stride, stride), (k // 2, k // 2), (1, 1), 1)), 8, 9)
    oh, ow = ref.shape[2:]
    res = None
    if residual:
        r = synth.tensor(cid, "r", ref.shape, -127, 127)
        ref = oracle.cvm_right_shift(oracle.relu(oracle.elemwise("elemwise_add", ref, r)), 8, 1)
        res = hipops.pack_act_i8(T(r, dev))
    out = hipops.conv2d_i8(hipops.pack_act_i8(T(x, dev)), n, ic, h, w, hipops.pack_weights(T(wt, dev)), oc, k, k, T(b, dev),
                           hipops.chain(("relu",), ("cvm_right_shift", 8, 9)), res,
                           hipops.chain(("relu",), ("cvm_right_shift", 8, 1)) if residual else None,
                           out_is_i8=True, strides=(stride, stride), padding=(k // 2, k // 2))
    got = hipops.unpack_act_i8(out, n, oc, oh, ow)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("n,ic,h,w,oc", [
    (9, 64, 32, 32, 256),     # whole tiles of pixels
    (11, 64, 30, 30, 200),    # pixels and channels that end inside a tile
])
@pytest.mark.parametrize("multiply", [False, True])
def test_tile_128_by_128_with_a_fused_pool(n, ic, h, w, oc, multiply, dev, tile):
    cid = "tile128-pool-%d" % n
    x = synth.tensor(cid, "x", (n, ic, h, w), -127, 127)
    wt = synth.tensor(cid, "w", (oc, ic, 3, 3), -127, 127)
    b = synth.tensor(cid, "b", (oc,), -32768, 32768)
    v = oracle.conv2d(x, wt, b, (1, 1), (1, 1), (1, 1), 1)
    chain = [("cvm_right_shift", 8, 9)]
    if multiply:   # a chain that falls as its input grows: the maximum comes behind it
        v, chain = -3 * v, [("mul", -3), ("cvm_right_shift", 8, 11)]
    ref = oracle.max_pool2d(oracle.cvm_right_shift(v, *chain[-1][1:]), (2, 2), (2, 2), (0, 0), False)
    out = hipops.conv2d_pool2_i8(hipops.pack_act_i8(T(x, dev)), n, ic, h, w, hipops.pack_weights(T(wt, dev)), oc, 3, 3, T(b, dev),
                                 hipops.chain(*chain), padding=(1, 1))
    got = hipops.unpack_act_i8(out, n, oc, h // 2, w // 2)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("n,ic,hw,oc,k,takes", [
    (9, 256, 32, 256, 3, "big cfg 3"),      # 144 tiles of 128 x 128, K = 2304
    (9, 224, 32, 256, 3, "wave"),           # K = 2016
    (9, 256, 31, 256, 3, "wave"),           # 136 tiles
    (9, 1024, 32, 256, 1, "big cfg 3"),     # K = 1024 and 9 MiB of input
    (4, 1024, 32, 640, 1, "wave"),          # 160 tiles, 4 MiB
    (18, 1024, 32, 256, 1, "big cfg 1"),    # 144 tiles of 128 x 256
    (18, 512, 32, 256, 1, "wave"),          # K = 512 and 9 MiB
    (36, 512, 32, 128, 1, "big cfg 1"),     # 18 MiB
    (20, 512, 32, 256, 1, "big cfg 1"),     # 160 tiles
])
def test_which_layers_take_the_large_tiles(n, ic, hw, oc, k, takes, dev, monkeypatch):
    gen = torch.Generator(device=dev)
    gen.manual_seed(ic)
    xp = hipops.pack_act_i8(torch.randint(-127, 128, (n, ic, hw, hw), dtype=torch.int32, device=dev, generator=gen))
    wp = hipops.pack_weights(torch.randint(-127, 128, (oc, ic, k, k), dtype=torch.int32, device=dev, generator=gen))

    def run():
        return hipops.conv2d_i8(xp, n, ic, hw, hw, wp, oc, k, k, None, hipops.chain(("cvm_right_shift", 8, 10)), padding=(k // 2, k // 2))
    lib().cvmhip_kernel_timing_begin()
    out = run()
    torch.cuda.synchronize()
    buf = ctypes.create_string_buffer(1 << 16)
    check(lib().cvmhip_kernel_timing_end_launches(buf, len(buf)))
    assert takes in str(json.loads(buf.value.decode())[-1])
    monkeypatch.setenv("CVM_HIP_CONV", "wave")
    assert torch.equal(out, run())


@pytest.mark.parametrize("n,h,w,oc,pool,lo,hi,shift,takes", [
    (16, 16, 32, 640, False, -508, 508, 2, True),     # whole patches
    (16, 16, 32, 640, True, -508, 508, 2, True),
    (4, 50, 96, 256, False, 0, 127, 0, True),         # the last row of patches ends inside; 16 rows of 32
    (4, 50, 96, 256, True, 0, 127, 0, True),
    (6, 40, 59, 320, False, -128, 127, 0, True),      # 8 rows of 64, a column of pixels past the image
    (6, 40, 58, 320, True, -2048, 2047, 4, True),
    (11, 127, 161, 128, False, -127, 127, 0, True),   # several patches to a workgroup, odd extents
    (11, 126, 162, 128, True, -127, 127, 0, True),
    (16, 28, 28, 320, False, -127, 127, 0, False),    # 160 workgroups, 490 tiles of 64 x 128
    (16, 28, 28, 320, True, -127, 127, 0, True),      # with the pool
    (25, 28, 28, 192, False, -127, 127, 0, False),    # 150 workgroups, 462 tiles of 64 x 128, 154 of 128 x 256
    (26, 28, 28, 192, False, -127, 127, 0, True),     # 160 of 128 x 256
    (84, 28, 28, 64, False, -127, 127, 0, True),      # 515 tiles of 64 x 128
    (83, 28, 28, 64, False, -127, 127, 0, False),     # 509
    (37, 16, 32, 256, False, -127, 127, 0, False),    # 148 workgroups
    (64, 33, 48, 128, False, -127, 127, 0, False),    # patches of 1.6 times the image
    (16, 16, 32, 640, False, -512, 512, 2, False),    # 128 after the shift: its low byte
    (16, 16, 32, 608, False, -127, 127, 0, False),    # channels that are no multiple of 64
])
def test_filter_and_patch_in_lds(n, h, w, oc, pool, lo, hi, shift, takes, dev, monkeypatch):
    gen = torch.Generator(device=dev)
    gen.manual_seed(h * w)
    x = torch.randint(-4, 5, (n, 64, h, w), dtype=torch.int32, device=dev, generator=gen)
    wt = torch.randint(-9, 10, (oc, 64, 3, 3), dtype=torch.int32, device=dev, generator=gen)
    xp, wp = hipops.pack_act_i8(x), hipops.pack_weights(wt)
    b = torch.randint(-300, 300, (oc,), dtype=torch.int32, device=dev, generator=gen)
    chain = hipops.Chain()
    chain.count = 1
    chain.stage[0] = hipops.Stage(5, 0, shift, lo, hi)
    op = hipops.conv2d_pool2_i8 if pool else hipops.conv2d_i8

    def run():
        lib().cvmhip_kernel_timing_begin()
        out = op(xp, n, 64, h, w, wp, oc, 3, 3, b, chain, padding=(1, 1))
        torch.cuda.synchronize()
        buf = ctypes.create_string_buffer(1 << 16)
        check(lib().cvmhip_kernel_timing_end_launches(buf, len(buf)))
        size = (h // 2, w // 2) if pool else (h, w)
        return hipops.unpack_act_i8(out, n, oc, *size), "k_conv_halo" in str(json.loads(buf.value.decode())[-1])

    got, halo = run()
    assert halo == takes
    monkeypatch.setenv("CVM_HIP_CONV", "wave")
    want, halo = run()
    assert not halo and torch.equal(got, want)
    if h * w * oc < 400000:   # the last image against the oracle as well
        v = oracle.conv2d(x[n - 1:].cpu().numpy(), wt.cpu().numpy(), b.cpu().numpy(), (1, 1), (1, 1), (1, 1), 1)
        v = (np.clip(v, lo, hi) >> shift).astype(np.int8).astype(np.int32)
        if pool:
            v = oracle.max_pool2d(v, (2, 2), (2, 2), (0, 0), False)
        assert np.array_equal(got[n - 1:].cpu().numpy(), v)

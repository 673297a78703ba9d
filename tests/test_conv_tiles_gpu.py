"""Large-tile convolution kernel with the 128 x 128 tile, which the dispatch takes for layers of too few pixels for the
128 x 256 one: edges of its range, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from cvm_runtime_amd import hipops, synth

pytestmark = pytest.mark.gpu


def T(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(dev)


@pytest.mark.parametrize("n,ic,h,w,oc,k,stride,residual", [
    (9, 64, 32, 32, 256, 3, 1, False),     # 144 tiles: the least that takes it
    (11, 512, 29, 29, 200, 1, 1, True),    # pixels and channels that end inside a tile, shortest K, residual
    (47, 96, 28, 28, 130, 3, 2, False),    # two channels in the last tile, K of 864
])
def test_tile_128_by_128(n, ic, h, w, oc, k, stride, residual, dev):
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

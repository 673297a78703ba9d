"""Non-maximum suppression at the edges of its split: windows of rows, kept rows beyond the LDS list, classes sharing a
workgroup, the ranking's slices and chunks -- against the oracle, output and mutated input."""
import numpy as np
import pytest
import torch

import oracle
from cvm_runtime_amd import hipops, synth

pytestmark = pytest.mark.gpu


def _rows(cid, b, n, ids, extent, side, apart):
    x = np.zeros((b, n, 6), np.int32)
    x[:, :, 0] = synth.tensor(cid, "id", (b, n), ids[0], ids[1])
    x[:, :, 1] = synth.tensor(cid, "score", (b, n), -127, 127)
    if apart:   # a grid of boxes that never meet: every row is kept
        at = np.arange(n)
        x[:, :, 2], x[:, :, 3] = (at % 64) * 2 * side, (at // 64) * 2 * side
    else:
        x[:, :, 2:4] = synth.tensor(cid, "xy", (b, n, 2), 0, extent)
    x[:, :, 4:6] = x[:, :, 2:4] + 1 + synth.tensor(cid, "wh", (b, n, 2), side // 2, side)
    return x


@pytest.mark.parametrize("b,n,ids,extent,side,apart,force,top_k,keep", [
    (1, 1, (0, 0), 64, 16, False, False, -1, -1),
    (2, 33, (0, 1), 64, 16, False, True, -1, -1),
    (1, 64, (0, 0), 64, 16, False, False, 63, -1),
    (1, 1025, (-1, 200), 256, 32, False, False, -1, 7),       # ids that share a class, one row past a window
    (2, 2050, (0, 0), 0, 16, True, False, -1, 2049),          # more kept rows than the LDS list holds
    (1, 3200, (-1, 60), 0, 16, True, True, -1, -1),           # the same with cuts at negative ids
    (1, 2300, (0, 0), 1 << 29, 1 << 24, False, True, -1, -1), # boxes whose products need 64 bits
    (1, 8193, (0, 80), 512, 64, False, False, 8191, -1),      # one row past a chunk of the ranking
    (1, 32767, (0, 80), 2048, 64, False, False, 1000, 100),
    (1, 32768, (0, 80), 2048, 64, False, False, 1000, 100),   # ranked by the sort
])
def test_nms_splits(b, n, ids, extent, side, apart, force, top_k, keep, dev):
    x = _rows("nms-split-%d-%d" % (n, top_k), b, n, ids, extent, side, apart)
    vc = np.full((b,), n, np.int32)
    init = np.full_like(x, 5)
    y_ref, x_after = oracle.non_max_suppression(x, vc, 45, force, top_k, max_output_size=keep, y_init=init)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    tx, ty = T(x), T(init)
    hipops.non_max_suppression(tx, T(vc), ty, 45, force, top_k, max_output_size=keep)
    assert np.array_equal(ty.cpu().numpy(), y_ref) and np.array_equal(tx.cpu().numpy(), x_after)

"""Non-maximum suppression at the edges of its split: windows of rows, kept rows beyond the LDS list, classes sharing a
workgroup, the ranking's slices and chunks -- against the oracle, output and mutated input."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from cvm_runtime_amd import check, hipops, lib, synth

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


@pytest.mark.parametrize("b,n,ids,coords,force", [
    (1, 128, 1, 100, True), (1, 129, 1, 100, True),            # the least number of rows for the masks, one below it
    (1, 1024, 1, 400, True), (1, 1025, 1, 400, True),          # the most, one above it
    (4, 961, 1, 400, True),
    (1, 8200, 20, 2000, False), (2, 8192, 40, 2000, False),    # several workgroups to a class
    (3, 600, 1, 200, True), (5, 400, 1, 200, True),
    (1, 700, 2, 300, False),                                   # two ids that share a class
    (1, 640, 1, 16384, True), (1, 640, 1, 16385, True),        # coordinates at the edge of 15 bits, one beyond it
])
def test_nms_pairs(b, n, ids, coords, force, dev):
    """Classes of as many rows as the walk tests by masks, boxes with coordinates of both signs; with the caller's workspace and with
    the static one, which has no room for masks."""
    cid = "nms-pairs-%d-%d-%d" % (b, n, coords)
    x = np.zeros((b, n, 6), np.int32)
    x[:, :, 0] = synth.tensor(cid, "id", (b, n), 0, ids - 1) * (64 if ids == 2 else 1)
    x[:, :, 1] = synth.tensor(cid, "score", (b, n), -127, 127)
    x[:, :, 2:4] = synth.tensor(cid, "xy", (b, n, 2), -coords, coords - 1 - 64)
    x[:, :, 4:6] = x[:, :, 2:4] + synth.tensor(cid, "wh", (b, n, 2), -2, 64)   # some empty
    x[:, 0, 2:6] = (-coords, -coords, -coords + 70, -coords + 70)
    x[:, 1, 2:6] = (coords - 71, coords - 71, coords - 1, coords - 1)
    x[:, 2:40, 2:6] = x[:, :2, 2:6].repeat(19, 1) + synth.tensor(cid, "near", (b, 38, 4), 0, 1) * [1, 1, 0, 0]
    vc = np.full((b,), n, np.int32)
    init = np.full_like(x, 5)
    y_ref, x_after = oracle.non_max_suppression(x, vc, 30, force, -1, max_output_size=-1, y_init=init)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    for call in (hipops.non_max_suppression, hipops.non_max_suppression_static):
        tx, ty = T(x), T(init)
        call(tx, T(vc), ty, 30, force, -1, max_output_size=-1)
        assert np.array_equal(ty.cpu().numpy(), y_ref) and np.array_equal(tx.cpu().numpy(), x_after)


@pytest.mark.parametrize("n,k", [(1, 6), (255, 6), (257, 2), (8192, 6), (8193, 6), (300, 8), (300, 9)])   # one launch up to 8192; rows in registers up to 8
def test_valid_counts_splits(n, k, dev):
    x = synth.tensor("gvc", "%d-%d" % (n, k), (2, n, k), -127, 127)
    vc, y = hipops.get_valid_counts(torch.from_numpy(x).to(dev), 20)
    for b in range(2):
        rows = x[b][x[b][:, 1] > 20]
        assert int(vc[b]) == len(rows)
        got = y[b].cpu().numpy()
        assert np.array_equal(got[:len(rows)], rows) and (got[len(rows):] == -1).all()


@pytest.mark.parametrize("b,n,ids,force,top_k", [
    (2, 5000, 20, False, 128), (2, 5000, 1, False, 129),      # the masks begin at 129 candidates
    (2, 5000, 1, True, 400), (3, 1100, 1, False, 1024), (2, 8200, 8, False, 1000), (2, 1100, 1, False, -1), (2, 300, 2, False, 0),
])
def test_nms_workspace_of_a_top_k(b, n, ids, force, top_k, dev):
    """The walk stays inside a workspace that holds masks for top_k rows, and one byte less is refused."""
    x = _rows("nms-ws-%d-%d" % (n, top_k), b, n, (0, ids - 1), 512, 48, False)
    vc = np.full((b,), n, np.int32)
    init = np.full_like(x, 5)
    y_ref, x_after = oracle.non_max_suppression(x, vc, 45, force, top_k, max_output_size=-1, y_init=init)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    tx, tv, ty = T(x), T(vc), T(init)
    need = lib().cvmhip_nms_topk_workspace_bytes(b, n, 6, top_k)
    ws = torch.full((need + 65536,), 0x5a, dtype=torch.uint8, device=dev)

    def call(size):
        return lib().cvmhip_non_max_suppression(ctypes.c_void_p(tx.data_ptr()), ctypes.c_void_p(tv.data_ptr()), ctypes.c_void_p(ty.data_ptr()), b, n, 6, -1, 45,
                                                top_k, 2, 1, 0, int(force), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(size), None)
    assert call(need - 1) == 10
    torch.cuda.synchronize()
    check(call(need))
    torch.cuda.synchronize()
    assert np.array_equal(ty.cpu().numpy(), y_ref) and np.array_equal(tx.cpu().numpy(), x_after)
    assert bool((ws[need:] == 0x5a).all())

"""The calls of csrc/binding/hipops_native.cc through ctypes, for an installation whose torch comes without its C++ headers
(the binding cannot be compiled there).  Same arguments, same results, 5 us more of host time on a call."""
import ctypes

import torch

from . import check, lib
from .hipops import _conv_stream, _new, _ptr, _shape, _stream, _workspace, broadcast_shape, conv_out_hw, pool_out

_UNARY = ("relu", "cvm_clip", "cvm_right_shift", "cvm_left_shift", "clip", "abs", "negative", "cvm_precision")
_UNARY_ARGS = (0, 1, 2, 2, 2, 0, 0, 0)


def _size(t):
    return ctypes.c_size_t(t.numel())


def _scratch(t):
    return ctypes.c_void_p(t.data_ptr())


def unary(op, x, out, p, q):
    y = torch.empty_like(x) if out is None else out
    args = [ctypes.c_int32(v) for v in (p, q)[:_UNARY_ARGS[op]]]
    check(getattr(lib(), "cvmhip_" + _UNARY[op])(_ptr(x), _ptr(y), ctypes.c_int64(x.numel()), *args, _stream()))
    return y


def elemwise(op, a, b, out):
    c = torch.empty_like(a) if out is None else out
    check(lib().cvmhip_elemwise(op, _ptr(a), _ptr(b), _ptr(c), ctypes.c_int64(a.numel()), _stream()))
    return c


def broadcast(op, a, b):
    cs = broadcast_shape(a.shape, b.shape)
    c = _new(cs, a)
    check(lib().cvmhip_broadcast(op, _ptr(a), _shape(a.shape), a.dim(), _ptr(b), _shape(b.shape), b.dim(), _ptr(c), _shape(cs),
                                 len(cs), _stream()))
    return c


def conv2d(x, w, b, strides, padding, dilation, groups):
    n, ic, h, wd = x.shape
    oc, _, kh, kw = w.shape
    oh, ow = conv_out_hw(h, wd, kh, kw, strides[0], strides[1], padding[0], padding[1], dilation[0], dilation[1])
    y = _new((n, oc, oh, ow), x)
    ws = _workspace(lib().cvmhip_conv2d_workspace_bytes(n, ic, h, wd, oc, kh, kw, groups), x.device)
    check(lib().cvmhip_conv2d(_ptr(x), _ptr(w), _ptr(b), _ptr(y), n, ic, h, wd, oc, kh, kw, strides[0], strides[1], padding[0],
                              padding[1], dilation[0], dilation[1], groups, _scratch(ws), _size(ws), _conv_stream()))
    return y


def dense(x, w, b, operand_bits):
    m, k = x.shape
    n = w.shape[0]
    y = _new((m, n), x)
    ws = _workspace(lib().cvmhip_dense_workspace_bytes(m, k, n), x.device)
    check(lib().cvmhip_dense(_ptr(x), _ptr(w), _ptr(b), _ptr(y), m, k, n, operand_bits, _scratch(ws), _size(ws), _conv_stream()))
    return y


def max_pool2d(x, pool_size, strides, padding, ceil_mode):
    n, c, h, w = x.shape
    pad = list(padding) * 2 if len(padding) == 1 else padding
    oh = pool_out(h, pool_size[0], strides[0], pad[0], ceil_mode)
    ow = pool_out(w, pool_size[1], strides[1], pad[1], ceil_mode)
    y = _new((n, c, oh, ow), x)
    check(lib().cvmhip_max_pool2d(_ptr(x), _ptr(y), n, c, h, w, oh, ow, pool_size[0], pool_size[1], strides[0], strides[1], pad[0],
                                  pad[1], _stream()))
    return y


def reduce(op, x, shape, axes, exclude):
    y = _new(shape, x)
    check(lib().cvmhip_reduce(op, _ptr(x), _shape(x.shape), x.dim(), _ptr(y), ctypes.c_int64(y.numel()),
                              _shape(axes) if len(axes) else None, len(axes), exclude, _stream()))
    return y


def get_valid_counts(x, score_threshold):
    b, n, k = x.shape
    vc, y = _new((b,), x), torch.empty_like(x)
    ws = _workspace(lib().cvmhip_get_valid_counts_workspace_bytes(b, n), x.device)
    check(lib().cvmhip_get_valid_counts(_ptr(x), _ptr(vc), _ptr(y), b, n, k, score_threshold, _scratch(ws), _size(ws), _stream()))
    return vc, y


def non_max_suppression(x, valid_count, y, iou_threshold, force_suppress, top_k, id_index, coord_start, score_index, max_output_size):
    b, n, k = x.shape
    ws = _workspace(lib().cvmhip_nms_topk_workspace_bytes(b, n, k, top_k), x.device)
    check(lib().cvmhip_non_max_suppression(_ptr(x), _ptr(valid_count), _ptr(y), b, n, k, max_output_size, iou_threshold, top_k,
                                           coord_start, score_index, id_index, int(bool(force_suppress)), _scratch(ws), _size(ws),
                                           _stream()))
    return y

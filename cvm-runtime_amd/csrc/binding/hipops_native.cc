// Native half of hipops.py: the operators a node-by-node caller issues most, from torch tensors to the C ABI
// (include/cvm_hip_ops.h) in one Python call.
//
// What bounds them: such calls are 2-20 us of GPU work each, and the ctypes wrappers spent 6-7 us of host time on a call
// beside the launch itself (argument objects, two or three Python-level allocations, the stream object, reading three
// environment variables), so a node list of one image ran at the pace of the interpreter.  Here a call is argument
// checks, at::empty and the launch, about 1.5 us beside the launches.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <string>
#include <vector>

#include "../../../include/cvm_hip_ops.h"

namespace {

PyObject* g_error = nullptr;   // CvmHipError

struct Raised {};   // a Python exception is set

void Check(int rc) {
  if (rc == CVMHIP_OK) return;
  PyErr_Format(g_error, "cvmhip error %d: %s", rc, cvmhip_last_error());
  throw Raised();
}

// The C ABI's part of a call, without the interpreter's lock: a launch can block (a full queue), and other threads go on
// meanwhile.  Whatever can raise has been evaluated before.
template <typename F>
void Launch(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  Check(rc);
}

const at::Tensor& Any(PyObject* o) {
  if (!THPVariable_Check(o)) {
    PyErr_SetString(PyExc_AssertionError, "int32 contiguous CUDA tensor required");
    throw Raised();
  }
  return THPVariable_Unpack(o);
}

int32_t* Ptr(const at::Tensor& t) {
  if (!t.is_cuda() || t.scalar_type() != at::kInt || !t.is_contiguous()) {
    PyErr_SetString(PyExc_AssertionError, "int32 contiguous CUDA tensor required");
    throw Raised();
  }
  return static_cast<int32_t*>(t.data_ptr());
}

int32_t* Ptr(PyObject* o) { return o == Py_None ? nullptr : Ptr(Any(o)); }

long long Int(PyObject* o) {
  PyObject* i = PyNumber_Index(o);
  if (!i) throw Raised();
  const long long v = PyLong_AsLongLong(i);
  Py_DECREF(i);
  if (v == -1 && PyErr_Occurred()) throw Raised();
  return v;
}

std::vector<int64_t> Ints(PyObject* o, size_t least = 0) {
  PyObject* seq = PySequence_Fast(o, "a sequence of integers is required");
  if (!seq) throw Raised();
  std::vector<int64_t> v;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* e = PyNumber_Index(PySequence_Fast_GET_ITEM(seq, i));
    if (!e) break;
    v.push_back(PyLong_AsLongLong(e));
    Py_DECREF(e);
  }
  Py_DECREF(seq);
  if (PyErr_Occurred()) throw Raised();
  if (v.size() < least) {
    PyErr_SetString(PyExc_IndexError, "tuple index out of range");
    throw Raised();
  }
  return v;
}

void Dims(const at::Tensor& t, int nd) {
  if (t.dim() == nd) return;
  PyErr_Format(PyExc_ValueError, "a tensor of %d dimensions is required, got %d", nd, static_cast<int>(t.dim()));
  throw Raised();
}

at::Tensor New(at::IntArrayRef shape, const at::Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(at::kInt).device(like.device()));
}

// scratch from torch's allocator, which aligns to 512 bytes
at::Tensor Scratch(size_t bytes, const at::Tensor& like) {
  return at::empty({static_cast<int64_t>(bytes < 256 ? 256 : bytes)}, at::TensorOptions().dtype(at::kByte).device(like.device()));
}

void* Stream() { return c10::hip::getCurrentHIPStream().stream(); }

// the test hooks of hipops._apply_conv_tuning
void ApplyConvTuning() {
  const char* kind = std::getenv("CVM_HIP_CONV");
  const char* cfg = std::getenv("CVM_HIP_WAVECFG");
  const char* tile = std::getenv("CVM_HIP_TILE");
  int k = 0, c = -1, wm = 0, wn = 0;
  if (kind) k = kind[0] == 'l' ? 1 : kind[0] == 'w' ? 2 : kind[0] == 'b' ? 3 : 0;
  if (cfg && cfg[0] >= '0' && cfg[0] <= '9') c = std::atoi(cfg);
  if (tile && std::string(tile).size() >= 3 && tile[1] == ',') {
    wm = tile[0] - '0';
    wn = tile[2] - '0';
  }
  Check(cvmhip_set_conv_tuning(k, c, wm, wn));
}

int64_t FloorDiv(int64_t a, int64_t b) {
  if (b == 0) {
    PyErr_SetString(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    throw Raised();
  }
  const int64_t q = a / b;
  return q * b != a && (a < 0) != (b < 0) ? q - 1 : q;
}

// ---- operators: each takes the arguments of its wrapper in hipops.py, in order
PyObject* Unary(PyObject* const* a) {
  const at::Tensor& x = Any(a[1]);
  int32_t* xp = Ptr(x);
  at::Tensor y = a[2] == Py_None ? at::empty_like(x) : Any(a[2]);
  int32_t* yp = Ptr(y);
  const int64_t n = x.numel();
  const int p = static_cast<int>(Int(a[3])), q = static_cast<int>(Int(a[4]));
  void* s = Stream();
  const long long op = Int(a[0]);
  Launch([&] {
    switch (op) {
      case 0: return cvmhip_relu(xp, yp, n, s);
      case 1: return cvmhip_cvm_clip(xp, yp, n, p, s);
      case 2: return cvmhip_cvm_right_shift(xp, yp, n, p, q, s);
      case 3: return cvmhip_cvm_left_shift(xp, yp, n, p, q, s);
      case 4: return cvmhip_clip(xp, yp, n, p, q, s);
      case 5: return cvmhip_abs(xp, yp, n, s);
      case 6: return cvmhip_negative(xp, yp, n, s);
      case 7: return cvmhip_cvm_precision(xp, yp, n, s);
    }
    return static_cast<int>(CVMHIP_ERR_ARG);
  });
  return THPVariable_Wrap(std::move(y));
}

PyObject* Elemwise(PyObject* const* a) {
  const at::Tensor &x = Any(a[1]), &y = Any(a[2]);
  at::Tensor z = a[3] == Py_None ? at::empty_like(x) : Any(a[3]);
  const int op = static_cast<int>(Int(a[0]));
  const int32_t *xp = Ptr(x), *yp = Ptr(y);
  int32_t* zp = Ptr(z);
  void* s = Stream();
  Launch([&] { return cvmhip_elemwise(op, xp, yp, zp, x.numel(), s); });
  return THPVariable_Wrap(std::move(z));
}

PyObject* Broadcast(PyObject* const* a) {
  const at::Tensor &x = Any(a[1]), &y = Any(a[2]);
  const int nd = static_cast<int>(std::max(x.dim(), y.dim()));
  std::vector<int64_t> shape(nd);
  for (int i = 0; i < nd; ++i) {
    const int64_t dx = i - (nd - x.dim()), dy = i - (nd - y.dim());
    shape[i] = std::max<int64_t>(dx >= 0 ? x.size(dx) : 1, dy >= 0 ? y.size(dy) : 1);
  }
  at::Tensor z = New(shape, x);
  const int op = static_cast<int>(Int(a[0]));
  const int32_t *xp = Ptr(x), *yp = Ptr(y);
  int32_t* zp = Ptr(z);
  void* s = Stream();
  Launch([&] {
    return cvmhip_broadcast(op, xp, x.sizes().data(), static_cast<int>(x.dim()), yp, y.sizes().data(), static_cast<int>(y.dim()), zp,
                            shape.data(), nd, s);
  });
  return THPVariable_Wrap(std::move(z));
}

PyObject* Conv2d(PyObject* const* a) {
  const at::Tensor &x = Any(a[0]), &w = Any(a[1]);
  Dims(x, 4);
  Dims(w, 4);
  const auto st = Ints(a[3], 2), pd = Ints(a[4], 2), dl = Ints(a[5], 2);
  const int groups = static_cast<int>(Int(a[6]));
  const int n = static_cast<int>(x.size(0)), ic = static_cast<int>(x.size(1)), h = static_cast<int>(x.size(2)), wd = static_cast<int>(x.size(3));
  const int oc = static_cast<int>(w.size(0)), kh = static_cast<int>(w.size(2)), kw = static_cast<int>(w.size(3));
  const int64_t oh = FloorDiv(h + 2 * pd[0] - (dl[0] * (kh - 1) + 1), st[0]) + 1;
  const int64_t ow = FloorDiv(wd + 2 * pd[1] - (dl[1] * (kw - 1) + 1), st[1]) + 1;
  at::Tensor y = New({n, oc, oh, ow}, x);
  at::Tensor ws = Scratch(cvmhip_conv2d_workspace_bytes(n, ic, h, wd, oc, kh, kw, groups), x);
  ApplyConvTuning();
  const int32_t *xp = Ptr(x), *wp = Ptr(w), *bp = Ptr(a[2]);
  int32_t* yp = Ptr(y);
  void* s = Stream();
  Launch([&] {
    return cvmhip_conv2d(xp, wp, bp, yp, n, ic, h, wd, oc, kh, kw, static_cast<int>(st[0]), static_cast<int>(st[1]),
                         static_cast<int>(pd[0]), static_cast<int>(pd[1]), static_cast<int>(dl[0]), static_cast<int>(dl[1]), groups,
                         ws.data_ptr(), static_cast<size_t>(ws.numel()), s);
  });
  return THPVariable_Wrap(std::move(y));
}

PyObject* Dense(PyObject* const* a) {
  const at::Tensor &x = Any(a[0]), &w = Any(a[1]);
  Dims(x, 2);
  const int m = static_cast<int>(x.size(0)), k = static_cast<int>(x.size(1)), n = static_cast<int>(w.size(0));
  at::Tensor y = New({m, n}, x);
  at::Tensor ws = Scratch(cvmhip_dense_workspace_bytes(m, k, n), x);
  ApplyConvTuning();
  const int32_t *xp = Ptr(x), *wp = Ptr(w), *bp = Ptr(a[2]);
  int32_t* yp = Ptr(y);
  const int bits = static_cast<int>(Int(a[3]));
  void* s = Stream();
  Launch([&] { return cvmhip_dense(xp, wp, bp, yp, m, k, n, bits, ws.data_ptr(), static_cast<size_t>(ws.numel()), s); });
  return THPVariable_Wrap(std::move(y));
}

PyObject* MaxPool2d(PyObject* const* a) {
  const at::Tensor& x = Any(a[0]);
  Dims(x, 4);
  const auto k = Ints(a[1], 2), st = Ints(a[2], 2);
  auto pd = Ints(a[3], 1);
  if (pd.size() == 1) pd.push_back(pd[0]);
  const int ceil = PyObject_IsTrue(a[4]);
  if (ceil < 0) throw Raised();
  const int64_t h = x.size(2), w = x.size(3);
  const int64_t oh = FloorDiv(h + 2 * pd[0] - k[0] + (ceil ? st[0] - 1 : 0), st[0]) + 1;
  const int64_t ow = FloorDiv(w + 2 * pd[1] - k[1] + (ceil ? st[1] - 1 : 0), st[1]) + 1;
  at::Tensor y = New({x.size(0), x.size(1), oh, ow}, x);
  auto i = [](int64_t v) { return static_cast<int>(v); };
  const int32_t* xp = Ptr(x);
  int32_t* yp = Ptr(y);
  void* s = Stream();
  Launch([&] {
    return cvmhip_max_pool2d(xp, yp, i(x.size(0)), i(x.size(1)), i(h), i(w), i(oh), i(ow), i(k[0]), i(k[1]), i(st[0]), i(st[1]),
                             i(pd[0]), i(pd[1]), s);
  });
  return THPVariable_Wrap(std::move(y));
}

// op, x, output shape (hipops.reduce_shape), axes, exclude
PyObject* Reduce(PyObject* const* a) {
  const at::Tensor& x = Any(a[1]);
  const auto ys = Ints(a[2]), ax = Ints(a[3]);
  at::Tensor y = New(ys, x);
  const int op = static_cast<int>(Int(a[0])), exclude = static_cast<int>(Int(a[4]));
  const int32_t* xp = Ptr(x);
  int32_t* yp = Ptr(y);
  void* s = Stream();
  Launch([&] {
    return cvmhip_reduce(op, xp, x.sizes().data(), static_cast<int>(x.dim()), yp, y.numel(), ax.empty() ? nullptr : ax.data(),
                         static_cast<int>(ax.size()), exclude, s);
  });
  return THPVariable_Wrap(std::move(y));
}

PyObject* GetValidCounts(PyObject* const* a) {
  const at::Tensor& x = Any(a[0]);
  Dims(x, 3);
  const int b = static_cast<int>(x.size(0)), n = static_cast<int>(x.size(1)), k = static_cast<int>(x.size(2));
  at::Tensor vc = New({b}, x), y = at::empty_like(x);
  at::Tensor ws = Scratch(cvmhip_get_valid_counts_workspace_bytes(b, n), x);
  const int32_t* xp = Ptr(x);
  int32_t *cp = Ptr(vc), *yp = Ptr(y);
  const int32_t threshold = static_cast<int32_t>(Int(a[1]));
  void* s = Stream();
  Launch([&] { return cvmhip_get_valid_counts(xp, cp, yp, b, n, k, threshold, ws.data_ptr(), static_cast<size_t>(ws.numel()), s); });
  PyObject* v = THPVariable_Wrap(std::move(vc));
  PyObject* r = THPVariable_Wrap(std::move(y));
  PyObject* t = PyTuple_Pack(2, v, r);
  Py_DECREF(v);
  Py_DECREF(r);
  return t;
}

// x, valid_count, y, iou, force, top_k, id_index, coord_start, score_index, max_output_size
PyObject* NonMaxSuppression(PyObject* const* a) {
  const at::Tensor& x = Any(a[0]);
  Dims(x, 3);
  const int b = static_cast<int>(x.size(0)), n = static_cast<int>(x.size(1)), k = static_cast<int>(x.size(2));
  int v[7];
  for (int i = 0; i < 7; ++i) v[i] = i == 1 ? PyObject_IsTrue(a[4]) : static_cast<int>(Int(a[3 + i]));
  at::Tensor ws = Scratch(cvmhip_nms_topk_workspace_bytes(b, n, k, v[2]), x);
  int32_t *xp = Ptr(x), *cp = Ptr(a[1]), *yp = Ptr(a[2]);
  void* s = Stream();
  Launch([&] {
    return cvmhip_non_max_suppression(xp, cp, yp, b, n, k, v[6], v[0], v[2], v[4], v[5], v[3], v[1], ws.data_ptr(),
                                      static_cast<size_t>(ws.numel()), s);
  });
  Py_INCREF(a[2]);
  return a[2];
}

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* Entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments are required, got %d", N, static_cast<int>(n));
    return nullptr;
  }
  try {
    return F(args);
  } catch (const Raised&) {
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

PyObject* Setup(PyObject*, PyObject* error) {
  Py_INCREF(error);
  g_error = error;
  Py_RETURN_NONE;
}

#define METHOD(name, fn, n) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<fn, n>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {METHOD("unary", Unary, 5),
                          METHOD("elemwise", Elemwise, 4),
                          METHOD("broadcast", Broadcast, 3),
                          METHOD("conv2d", Conv2d, 7),
                          METHOD("dense", Dense, 4),
                          METHOD("max_pool2d", MaxPool2d, 5),
                          METHOD("reduce", Reduce, 5),
                          METHOD("get_valid_counts", GetValidCounts, 2),
                          METHOD("non_max_suppression", NonMaxSuppression, 10),
                          {"setup", Setup, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_hipops_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hipops_native() { return PyModule_Create(&kModule); }

"""MI355X (gfx950) backend for the CVM deterministic integer inference path.

The product is the shared library `libcvm_runtime_hip.so` built from csrc/:
hand-written HIP kernels behind the operator-level C ABI
(include/cvm_hip_ops.h) and a C++ graph runtime behind the reference's model
C API (include/cvm_c_api.h).  This Python package is only a loader plus thin
wrappers (ctypes, and csrc/binding for the operators a node-by-node caller issues
most); torch is used for device memory and streams, nothing else.

There is no CPU fallback: if the library is missing or no GPU is present the
wrappers raise.
"""
import ctypes
import os
import warnings

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libcvm_runtime_hip.so")
NATIVE_PATH = os.path.join(_HERE, "_hipops_native.so")
_lib = None
_native = None


class CvmHipError(RuntimeError):
    pass


def lib():
    """The loaded shared library (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise CvmHipError(
                "%s is missing: build it with `python cvm-runtime_amd/build.py` "
                "(there is no CPU fallback)" % LIB_PATH)
        _lib = ctypes.CDLL(LIB_PATH)
        _lib.cvmhip_last_error.restype = ctypes.c_char_p
        for name in ("cvmhip_conv2d_workspace_bytes", "cvmhip_dense_workspace_bytes",
                     "cvmhip_get_valid_counts_workspace_bytes", "cvmhip_nms_workspace_bytes", "cvmhip_nms_topk_workspace_bytes",
                     "cvmhip_nms_static_capacity_bytes",
                     "cvmhip_packed_weight_bytes", "cvmhip_packed_act_bytes", "cvmhip_packed_depthwise_bytes"):
            getattr(_lib, name).restype = ctypes.c_size_t
    return _lib


def native():
    """The native half of hipops.py; hipops_plain, with a warning, where the build had to leave it out."""
    global _native
    if _native is None:
        lib()
        if not os.path.exists(NATIVE_PATH):
            warnings.warn("%s is missing: operator calls go through ctypes and take 5 us more each" % NATIVE_PATH)
            from . import hipops_plain
            _native = hipops_plain
            return _native
        import importlib.util
        import torch  # noqa: F401  (its libraries are what the module links to)
        spec = importlib.util.spec_from_file_location("_hipops_native", NATIVE_PATH)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.setup(CvmHipError)
        _native = mod
    return _native


def check(rc):
    if rc != 0:
        raise CvmHipError("cvmhip error %d: %s" % (rc, lib().cvmhip_last_error().decode()))

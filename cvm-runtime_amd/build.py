"""Build the gfx950 shared library in-tree: python cvm-runtime_amd/build.py

Every .hip / .cc file under csrc/ is compiled with hipcc for gfx950 and linked
into cvm-runtime_amd/libcvm_runtime_hip.so, the one library that exports both
the operator-level C ABI (include/cvm_hip_ops.h) and the model-level C ABI
(include/cvm_c_api.h).  csrc/binding/ becomes _hipops_native.so, the native half of
hipops.py; it is the only object that knows torch, and the library does not need it: without
torch's headers it is left out, and hipops goes through ctypes.
"""
import glob
import importlib.util
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libcvm_runtime_hip.so")
BINDING = os.path.join(HERE, "_hipops_native.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON = ["-O3", "-fPIC", "-std=c++17", "-fsigned-char", "-fvisibility=hidden", "-I" + os.path.join(HERE, "..", "include")]
# extra preprocessor definitions for a measurement build, e.g. CVM_HIP_DEFINES="-DCVM_SEQ_STAMPS"
COMMON += os.environ.get("CVM_HIP_DEFINES", "").split()
# packed-fp32 code generation is switched off for all device code
DEVICE = ["--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _compile(src):
    rel = os.path.relpath(src, CSRC).replace(os.sep, "_")
    obj = os.path.join(OBJ, rel + ".o")
    cmd = [HIPCC] + COMMON + (DEVICE if src.endswith(".hip") else ["-x", "c++"]) + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError("compile failed: %s\n%s" % (" ".join(cmd), out))
    if out.strip():
        sys.stderr.write(out + "\n")
    return obj


def _build_binding():
    """The binding, where torch is installed with its headers; the library does without, and hipops then uses ctypes."""
    if os.path.exists(BINDING):
        os.remove(BINDING)   # never one that belongs to another build of the library
    spec = importlib.util.find_spec("torch")
    torch = os.path.dirname(spec.origin) if spec else ""
    python = sysconfig.get_paths()["include"]
    for need in (os.path.join(torch, "include", "torch", "csrc", "autograd", "python_variable.h"),
                 os.path.join(torch, "include", "c10", "hip", "HIPStream.h"), os.path.join(python, "Python.h")):
        if not os.path.exists(need):
            sys.stderr.write("no %s: %s is left out\n" % (os.path.basename(need), os.path.basename(BINDING)))
            return
    inc = [os.path.join(torch, "include"), os.path.join(torch, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include"), python]
    cmd = ([HIPCC, "-O2", "-fPIC", "-shared", "-std=c++17", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM", "-x", "c++"] +
           ["-I" + d for d in inc] + [os.path.join(CSRC, "binding", "hipops_native.cc"), "-o", BINDING, "-L" + HERE,
            "-l:" + os.path.basename(LIB), "-L" + os.path.join(torch, "lib"), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10",
            "-lc10_hip", "-Wl,-rpath,$ORIGIN"])
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError("binding failed: %s\n%s" % (" ".join(cmd), r.stdout))


def build(verbose=False):
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "runtime", "*.cc")))
    with ThreadPoolExecutor(max_workers=8) as ex:
        objs = list(ex.map(_compile, srcs))
    cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=gfx950", "-o", LIB] + objs + ["-Wl,-Bsymbolic"]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout)
    _build_binding()
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)

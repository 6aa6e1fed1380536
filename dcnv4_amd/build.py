"""Builds libdcnv4_gfx950.so from dcnv4_amd/csrc/*.hip with hipcc, for gfx950 only, and the Python extension _native.so
(host code only: dcnv4_amd/csrc/binding/*.cpp, g++, against the installed torch and the library).

Takes the place of the reference's CUDAExtension build (DCNv4_op/setup.py:24-60): there is no
hipify pass and no torch extension machinery, just hipcc on hand-written HIP sources and a C ABI.
Usage: ``python dcnv4_amd/build.py [--force]`` (run as a script: importing the package needs the library).
"""
import concurrent.futures
import importlib.util
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "build")
LIB_PATH = os.path.join(HERE, "libdcnv4_gfx950.so")
SOURCES = ["capi.hip", "dcnv4_kernels.hip", "dcnv4_tiled_gather.hip", "dcnv4_window.hip", "dcnv4_grad_value.hip", "dcnv4_backward_dual.hip", "fda_kernels.hip", "fda_grad_value.hip",
           "depthwise_conv.hip", "layer_norm.hip", "center_feature.hip",
           "linear.hip", "linear_rows.hip", "linear_grad.hip", "mlp.hip", "conv.hip"]
HEADERS = [os.path.join(CSRC, "common.hpp"), os.path.join(CSRC, "mfma.hpp"), os.path.join(CSRC, "fragments.hpp"), os.path.join(CSRC, "dcnv4_at_once.hpp"), os.path.join(CSRC, "layer_norm.hpp"), os.path.join(CSRC, "linear.hpp"), os.path.join(CSRC, "conv.hpp"), os.path.join(CSRC, "launch.hpp"),
           os.path.join(CSRC, "dcnv4_tiled_gather.hpp"), os.path.join(CSRC, "dcnv4_window.hpp"), os.path.join(CSRC, "dcnv4_grad_value.hpp"),
           os.path.join(os.path.dirname(HERE), "include", "dcnv4_gfx950.h")]

BINDING = os.path.join(CSRC, "binding")
BINDING_SOURCES = ["module.cpp", "operators.cpp", "modules.cpp", "layers.cpp", "training.cpp", "attention.cpp", "convolutions.cpp"]
BINDING_HEADERS = [os.path.join(BINDING, "binding.hpp"), os.path.join(BINDING, "modules.hpp"), os.path.join(BINDING, "layers.hpp"),
                   os.path.join(CSRC, "linear.hpp"), os.path.join(CSRC, "conv.hpp"), os.path.join(CSRC, "layer_norm.hpp"),
                   os.path.join(os.path.dirname(HERE), "include", "dcnv4_gfx950.h")]
NATIVE_PATH = os.path.join(HERE, "_native.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")
# -packed-fp32-ops: keep the compiler from forming v_pk_*_f32 instructions.
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++20", "-fPIC", "-fno-gpu-rdc",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wall", "-Wno-pass-failed", "-Wno-unused-function", "-Wno-unknown-attributes"]


def _stale(target, deps):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def _torch_paths():
    spec = importlib.util.find_spec("torch")      # found, not imported
    return os.path.dirname(spec.origin)


def _run(cmd, what):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError("%s failed: %s\n%s" % (what, " ".join(cmd), err))
    if err.strip():
        sys.stderr.write(err + "\n")


def _compile(src, force):
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    path = os.path.join(CSRC, src)
    if force or _stale(obj, [path] + HEADERS):
        _run([HIPCC] + FLAGS + ["-c", path, "-o", obj], "hipcc")
    return obj


def _compile_binding(src, force):
    obj = os.path.join(OBJ_DIR, "binding_" + os.path.splitext(src)[0] + ".o")
    path = os.path.join(BINDING, src)
    if force or _stale(obj, [path] + BINDING_HEADERS):
        include = os.path.join(_torch_paths(), "include")
        _run([CXX, "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
              "-I" + include, "-I" + os.path.join(include, "torch", "csrc", "api", "include"), "-I/opt/rocm/include",
              "-I" + sysconfig.get_path("include"), "-c", path, "-o", obj], "g++")
    return obj


def build(force=False, verbose=True):
    os.makedirs(OBJ_DIR, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as pool:
        objs = [pool.submit(_compile, s, force) for s in SOURCES]
        binding = [pool.submit(_compile_binding, s, force) for s in BINDING_SOURCES]
        objs, binding = [f.result() for f in objs], [f.result() for f in binding]
    if force or _stale(LIB_PATH, objs):
        _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname,libdcnv4_gfx950.so", "-o", LIB_PATH] + objs, "link")
    if force or _stale(NATIVE_PATH, binding + [LIB_PATH]):
        lib = os.path.join(_torch_paths(), "lib")
        _run([CXX, "-shared", "-o", NATIVE_PATH] + binding + ["-L" + HERE, "-ldcnv4_gfx950", "-L" + lib, "-lc10", "-lc10_hip",
             "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,$ORIGIN"], "link")
    if verbose:
        print("built", LIB_PATH, "and", NATIVE_PATH)
    return LIB_PATH


if __name__ == "__main__":
    build(force="--force" in sys.argv)

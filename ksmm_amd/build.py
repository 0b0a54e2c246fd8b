"""Builds libksmm_hip.so for gfx950 with hipcc (cross-compiles without a GPU), and the CPython module
_native.so that KSLinear calls it through (that one needs g++ and PyTorch's headers; where it cannot be
built, a warning says why, and layers are launched through ctypes).

    python -m ksmm_amd.build          # rebuild everything
"""
import concurrent.futures
import os
import subprocess
import sys
import warnings

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libksmm_hip.so")
SOURCES = ["ksmm_api.hip", "ksmm_generic.hip", "ksmm_wave.hip", "ksmm_tile.hip", "ksmm_stream.hip", "ksmm_tile_bf.hip", "ksmm_rows_bf.hip", "ksmm_gemm.hip", "ksmm_split.hip", "ksmm_pair.hip", "ksmm_choose.hip", "ksmm_chain16.hip", "ksmm_chain16r.hip", "ksmm_transpose.hip", "ksmm_backward.hip", "ksmm_wgrad_bf.hip", "ksmm_wgrad_wide.hip", "ksmm_act_bwd.hip", "ksmm_quant.hip"]
# measurement aids of bench.py: a library of their own, outside the drop-in ABI
BENCH_LIB = os.path.join(HERE, "libksmm_bench.so")
BENCH_SOURCES = ["ksmm_probe.hip"]
# host side of KSLinear: a CPython module that links the library
NATIVE = os.path.join(HERE, "_native.so")
NATIVE_SOURCE = "ksmm_torch.cpp"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# packed fp32 VALU ops are switched off on purpose for this hardware
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", "-Wno-inline-asm",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _compile(src):
    obj = os.path.join(OBJ, src.replace(".hip", ".o"))
    cmd = [HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, r.stderr[-8000:]))
    noise = "is not a recognized feature for this target"
    warn = "\n".join(l for l in r.stderr.splitlines() if l.strip() and noise not in l)
    return obj, warn


def _compile_native():
    import sysconfig

    import torch

    root = os.path.dirname(torch.__file__)
    obj = os.path.join(OBJ, NATIVE_SOURCE.replace(".cpp", ".o"))
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           "/opt/rocm/include", sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), *("-I" + i for i in inc),
           "-c", os.path.join(CSRC, NATIVE_SOURCE), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed for %s:\n%s" % (NATIVE_SOURCE, r.stderr[-8000:]))
    return obj


def _link_native(obj):
    import torch

    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-shared", "-o", NATIVE, obj, LIB, "-L" + lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr[-4000:])


def build(verbose=False, jobs=8):
    os.makedirs(OBJ, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        native = ex.submit(_compile_native)
        results = list(ex.map(_compile, SOURCES + BENCH_SOURCES))
    objs = [o for o, _ in results[:len(SOURCES)]]
    bench_objs = [o for o, _ in results[len(SOURCES):]]
    if verbose:
        for _, w in results:
            if w:
                print(w, file=sys.stderr)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname,libksmm_hip.so", "-o", LIB] + objs,
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr[-4000:])
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", BENCH_LIB] + bench_objs,
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr[-4000:])
    try:
        _link_native(native.result())
    except (ImportError, OSError, RuntimeError) as e:
        if os.path.exists(NATIVE):
            os.remove(NATIVE)  # of an earlier build
        warnings.warn("%s is not built: %s" % (os.path.basename(NATIVE), e), RuntimeWarning)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))

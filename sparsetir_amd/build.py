"""Builds ``libsparsetir_amd.so`` (HIP kernels + C ABI) for gfx950 with hipcc, and ``_host.so``, the
native host path of the Python operators, against the installed torch.

Run as ``python -m sparsetir_amd.build``.  hipcc cross-compiles, so no GPU is needed.
The libraries are placed next to this file; they are what ``sparsetir_amd._lib`` and
``sparsetir_amd.ops`` load.
"""
import glob
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libsparsetir_amd.so")
HOST_SRC = os.path.join(CSRC, "bindings", "host.cpp")
HOST = os.path.join(HERE, "_host.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
          "-I", os.path.join(HERE, "..", "include")]
# Packed fp32 VALU ops are kept off for every device translation unit.
DEVICE = [f"--offload-arch={ARCH}", "-munsafe-fp-atomics",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# Per-file additions.  The destination-tiled RGMS kernel chains MFMAs through ordinary vector
# registers (one accumulator feeds the next stage's operand); with the accumulator-register form
# the compiler copies both accumulators between the two register files on every step.
EXTRA = {"rgms_tiles.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.cpp")))


def _build_host():
    """The extension module of the operators' host path; its link needs LIB."""
    import torch

    root = os.path.dirname(torch.__file__)
    libs = ["-L" + os.path.join(root, "lib"), "-L" + HERE, "-lsparsetir_amd", "-ltorch_python", "-ltorch_cpu", "-lc10",
            "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unused-parameter", "-DUSE_ROCM=1",
           "-D__HIP_PLATFORM_AMD__=1", "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch.compiled_with_cxx11_abi()),
           "-isystem", os.path.join(root, "include"),
           "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
           "-isystem", os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include"),
           "-isystem", sysconfig.get_paths()["include"], HOST_SRC, "-o", HOST] + libs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("building _host.so failed:\n" + r.stdout + r.stderr)
    return r.stdout + r.stderr


def _compile(src):
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    cmd = [HIPCC] + COMMON
    if src.endswith(".hip"):
        cmd += DEVICE + EXTRA.get(os.path.basename(src), []) + ["-x", "hip"]
    cmd += ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    return src, obj, r.returncode, r.stdout + r.stderr


def build(verbose=True, jobs=8):
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        results = list(ex.map(_compile, srcs))
    objs = []
    for src, obj, rc, log in results:
        log = "\n".join(l for l in log.splitlines()
                        if "packed-fp32-ops" not in l and "is not a recognized feature" not in l)
        if rc != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{log}")
        if verbose and log.strip():
            print(log)
        objs.append(obj)
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", LIB] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    log = _build_host()
    if verbose:
        if log.strip():
            print(log)
        print(f"built {LIB} from {len(srcs)} sources and {HOST}")
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)

"""Compile the package's native code, in-tree: the HIP sources under csrc/ for gfx950 into one C-ABI
shared library, and the host layer under csrc/host/ into a Python extension on top of it.

`python -m trainium_frontier_them_bones_amd.build` (or `build_library()`) runs hipcc on every
`csrc/*.hip` and the host compiler on every `csrc/host/*.cpp` in parallel and links `libtfb_hip.so`
and `_tfb_host.so` next to this file. hipcc cross-compiles, so no GPU is needed to build. The flags
switch packed-fp32 code generation off for device code.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_NAME = "libtfb_hip.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
HOST_SRC = os.path.join(CSRC, "host")
HOST_PATH = os.path.join(HERE, "_tfb_host.so")
OBJ_DIR = os.path.join(HERE, "build")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
] + os.environ.get("TFB_EXTRA_FLAGS", "").split()


CXX = os.environ.get("CXX", "g++")


def _host_flags():
    import torch
    from torch.utils.cpp_extension import include_paths
    inc = include_paths("cuda") + [sysconfig.get_paths()["include"]]
    return (["-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI] + ["-isystem" + p for p in inc],
            os.path.join(os.path.dirname(torch.__file__), "lib"))


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def host_sources():
    return sorted(f for f in os.listdir(HOST_SRC) if f.endswith(".cpp"))


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("%s failed:\n%s" % (what, r.stderr))
    return "\n".join(l for l in r.stderr.splitlines() if "not a recognized feature" not in l)


def _compile(src):
    obj = os.path.join(OBJ_DIR, src[:-4] + ".o")
    return obj, _run([HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj], "hipcc on " + src)


def _compile_host(src, flags):
    obj = os.path.join(OBJ_DIR, "host_" + src[:-4] + ".o")
    return obj, _run([CXX] + flags + ["-c", os.path.join(HOST_SRC, src), "-o", obj], CXX + " on " + src)


def build_library(verbose=True, jobs=None):
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs, hosts = sources(), host_sources()
    hflags, torch_lib = _host_flags()
    with ThreadPoolExecutor(max_workers=jobs or 8) as ex:
        host_jobs = [ex.submit(_compile_host, s, hflags) for s in hosts]   # (first: they take the longest)
        lib_jobs = [ex.submit(_compile, s) for s in srcs]
        objs, hobjs = [j.result() for j in lib_jobs], [j.result() for j in host_jobs]
    for (o, err), s in zip(objs + hobjs, srcs + hosts):
        if verbose and err.strip():
            print("[%s]\n%s" % (s, err), file=sys.stderr)
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-soname," + LIB_NAME, "-o", LIB_PATH] + [o for o, _ in objs], "link")
    _run([CXX, "-shared", "-o", HOST_PATH] + [o for o, _ in hobjs] + ["-L" + HERE, "-l:" + LIB_NAME, "-L" + torch_lib, "-lc10", "-lc10_hip",
         "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"], "link of the host layer")
    if verbose:
        print("built %s and %s from %d + %d sources" % (LIB_PATH, os.path.basename(HOST_PATH), len(srcs), len(hosts)))
    return LIB_PATH


if __name__ == "__main__":
    build_library()

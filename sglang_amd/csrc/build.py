"""Build libfp8k.so (hand-written HIP kernels for gfx950 + the C ABI) in-tree with hipcc, and _host.so (the native side of
the layer-level calls, a CPython extension over it) with the host compiler.

Usage: python sglang_amd/csrc/build.py [--force] [--jobs N]
Each .hip file is compiled to an object next to it and linked into sglang_amd/csrc/libfp8k.so.
"""
from __future__ import annotations

import argparse
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "libfp8k.so")
HOST_SRC = "host.cpp"
HOST = os.path.join(os.path.dirname(HERE), "_host.so")  # the extension module sglang_amd._host, linked against LIB
SOURCES = ["api.hip", "quant.hip", "gemm.hip", "moe.hip", "tune.hip"]
HEADERS = ["fp8k_common.h", "quant_math.h", "gemm_kernels.h", "gemm_direct.h", "gemm_direct_quant.h", "gemm_moe256.h", "gemm_moe_shortk.h", "gemm_skinny.h", "gemm_tile128.h", "gemm_tile64.h", "gemm_bmm.h", os.path.join("..", "..", "include", "fp8k.h"),
           os.path.join("..", "..", "include", "fp8k_tune.h")]

# -packed-fp32-ops off: packed float32 VALU forms are not used on this hardware pool.
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Wno-unknown-warning-option",
    "-Wno-pass-failed",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; the fp8k library can only be built with the ROCm toolchain")


def _stale(target: str, deps: list[str]) -> bool:
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.exists(d) and os.path.getmtime(d) > t for d in deps)


def _run(cmd: list[str]) -> None:
    p = subprocess.run(cmd, cwd=HERE, capture_output=True, text=True)
    err = "\n".join(l for l in (p.stdout + p.stderr).splitlines() if "not a recognized feature" not in l)
    if p.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), err))
    if err.strip():
        sys.stderr.write(err + "\n")


def _host_stale() -> bool:
    """Whether _host.so has to be built: older than its sources, or built for another torch, whose C++ interface it uses."""
    import torch

    if _stale(HOST, [os.path.join(HERE, HOST_SRC), os.path.abspath(__file__), os.path.join(HERE, "..", "..", "include", "fp8k.h")]):
        return True
    with open(HOST, "rb") as f:
        return _torch_mark(torch.__version__).encode() not in f.read()


def _torch_mark(version: str) -> str:
    return "built for torch %s;" % version


def _host_command() -> list[str]:
    """Host code only: the native side of the layer-level calls, against torch's C++ API."""
    import sysconfig

    import torch

    root = os.path.dirname(os.path.abspath(torch.__file__))
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"), "/opt/rocm/include",
           sysconfig.get_paths()["include"]]
    return [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
            "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), "-Wno-deprecated-declarations",
            '-DFP8K_TORCH_MARK="%s"' % _torch_mark(torch.__version__)] + [
        "-isystem" + d for d in inc] + [HOST_SRC, "-o", HOST, "-L" + HERE, "-lfp8k", "-L" + os.path.join(root, "lib"),
                                        "-ltorch_python", "-ltorch_hip", "-ltorch_cpu", "-ltorch", "-lc10_hip", "-lc10",
                                        "-Wl,-rpath,$ORIGIN/csrc"]


def build(force: bool = False, jobs: int = 4, verbose: bool = True) -> str:
    cc = hipcc()
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(HERE, s))]
    hdrs = [os.path.join(HERE, h) for h in HEADERS]
    objs = []
    todo = []
    for s in srcs:
        o = os.path.join(HERE, s[:-4] + ".o")
        objs.append(o)
        if force or _stale(o, [os.path.join(HERE, s), os.path.abspath(__file__)] + hdrs):
            todo.append([cc] + FLAGS + ["-c", s, "-o", o])
    if verbose and todo:
        print("[fp8k] compiling %d file(s) for gfx950" % len(todo), flush=True)
    with ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        list(ex.map(_run, todo))
    if todo or force or _stale(LIB, objs):
        _run([cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs)
        if verbose:
            print("[fp8k] linked", LIB, flush=True)
    if force or _host_stale():
        _run(_host_command())
        if verbose:
            print("[fp8k] linked", HOST, flush=True)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--jobs", type=int, default=4)
    a = ap.parse_args()
    build(force=a.force, jobs=a.jobs)

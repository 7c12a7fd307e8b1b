"""Compiles the HIP/C++ sources under ``relax_amd/csrc`` into ``librelax_amd_wq.so`` (gfx950), and
the calibration kernels (``calibrate.hip``: measurement only) into ``librelax_amd_wq_calibrate.so``.
These need no torch.  Where there is one, ``csrc/python/calls.cc`` becomes ``_calls.so`` for it.

hipcc cross-compiles without a GPU.  The library is built in-tree so that it
travels with the source tree to the machine that runs it.
"""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
if os.path.dirname(HERE) not in sys.path:
    sys.path.insert(0, os.path.dirname(HERE))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "librelax_amd_wq.so")
CALIBRATE_LIB = os.path.join(HERE, "librelax_amd_wq_calibrate.so")
CALIBRATE_SOURCES = ("calibrate.hip",)  # not linked into the product library
CALLS_SOURCE = os.path.join(CSRC, "python", "calls.cc")  # the linears of ops.py as a Python extension
CALLS_LIB = os.path.join(HERE, "_calls.so")
OBJDIR = os.path.join(HERE, "build")
CALLS_STAMP = os.path.join(OBJDIR, "_calls.torch")  # the version of torch that _calls.so was compiled for

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "--offload-arch=gfx950", "-fPIC", "-std=c++17", "-fvisibility=hidden",
    "-Wall", "-Wno-unused-function",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]

SOURCE_FLAGS = {"gemm_256.hip": ["-falign-loops=64"]}  # why: see that file


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".cc")))


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, *SOURCE_FLAGS.get(os.path.basename(src), ()), "-c", src, "-o", obj]
    if src.endswith(".cc"):
        cmd.insert(1, "-x")
        cmd.insert(2, "hip")
    p = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in p.stderr.splitlines() if "packed-fp32-ops" not in l)
    if p.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _torch_version():
    """The version of the installed torch, or None."""
    try:
        import torch
    except ImportError:
        return None
    return str(torch.__version__)


def _calls_stale() -> bool:
    if not os.path.exists(CALLS_LIB) or not os.path.exists(CALLS_STAMP):
        return True
    with open(CALLS_STAMP) as f:
        if f.read() != _torch_version():
            return True
    return any(os.path.getmtime(d) > os.path.getmtime(CALLS_LIB) for d in _deps(CALLS_SOURCE))


def _compile_calls() -> str:
    from torch.utils import cpp_extension

    dirs = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", f'-DRELAX_AMD_TORCH_VERSION="{_torch_version()}"', *(f"-I{d}" for d in dirs), CALLS_SOURCE,
           "-o", CALLS_LIB, *(f"-L{d}" for d in cpp_extension.library_paths()), "-lc10", "-ltorch_cpu", "-ltorch_python"]
    p = subprocess.run(cmd, capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError(f"g++ failed on {CALLS_SOURCE}:\n{p.stderr}")
    with open(CALLS_STAMP, "w") as f:
        f.write(_torch_version())
    return CALLS_LIB


def check_asm(name: str) -> None:
    from relax_amd import check_ring_asm

    check_ring_asm.check_source(HIPCC, [*(f for f in FLAGS if f != "-fPIC"), *SOURCE_FLAGS.get(name, ())], name)


def _deps(src: str, seen=None):
    """`src` and every file it includes with quotes, transitively."""
    seen = seen if seen is not None else set()
    if src in seen or not os.path.exists(src):
        return seen
    seen.add(src)
    with open(src) as f:
        for line in f:
            line = line.strip()
            if line.startswith('#include "'):
                _deps(os.path.normpath(os.path.join(os.path.dirname(src), line.split('"')[1])), seen)
    return seen


def _stale(src: str) -> bool:
    obj = os.path.join(OBJDIR, os.path.basename(src) + ".o")
    if not os.path.exists(obj):
        return True
    t = os.path.getmtime(obj)
    return any(os.path.getmtime(d) > t for d in _deps(src))


def build(verbose: bool = True, incremental: bool = False) -> str:
    """Compile every source (with `incremental`, only those newer than their object file, headers
    included) and link the shared library; returns its path."""
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    todo = [s for s in srcs if _stale(s)] if incremental else srcs
    from relax_amd import check_ring_asm

    # some kernels wait by hand for loads that the compiler does not see: the code generated for them is verified
    checked = [s for s in todo if os.path.basename(s) in check_ring_asm.SOURCES + check_ring_asm.HELD_SOURCES + check_ring_asm.DIRECT_LOAD_SOURCES]
    if todo:
        with concurrent.futures.ThreadPoolExecutor(max_workers=8) as ex:
            compiled = [ex.submit(_compile, s) for s in todo]
            checks = [ex.submit(check_asm, os.path.basename(s)) for s in checked]
            concurrent.futures.wait(compiled + checks)
            for f, s in zip(checks, checked):  # an incremental build must not take a refused object for up to date
                obj = os.path.join(OBJDIR, os.path.basename(s) + ".o")
                if f.exception() is not None and os.path.exists(obj):
                    os.remove(obj)
            for f in compiled + checks:
                f.result()
    for lib, want in ((LIB, False), (CALIBRATE_LIB, True)):
        objs = [os.path.join(OBJDIR, os.path.basename(s) + ".o") for s in srcs
                if (os.path.basename(s) in CALIBRATE_SOURCES) == want]
        subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib, *objs])
    # last: the libraries above are for programs without torch too
    if _torch_version() is None:
        print(f"no torch: {CALLS_LIB} is not built", flush=True)
    elif not incremental or _calls_stale():
        _compile_calls()
    if verbose:
        print(f"built {LIB}: compiled {len(todo)} of {len(srcs)} sources", flush=True)
    return LIB


if __name__ == "__main__":
    build(incremental="--incremental" in sys.argv)

"""Builds libqws.so (HIP, gfx950) in-tree, qwen-warp_amd/lib/libqws.so, and beside it the host packing module
_qws_hostpack.<ABI tag>.so (C++ over the CPython API, for the interpreter that runs the build; without a compiler or
Python headers the build warns and goes on, and id lists are packed in Python).

  python qwen-warp_amd/build.py

Each source is compiled to an object in parallel (no device code crosses files: every kernel is launched from its own
file, the shared device helpers are inline), then the objects are linked.  Flags: -ffp-contract=off (every
floating-point operation one IEEE rounding, as the CPU definition), no fast-math, packed fp32 instructions off
(-Xclang -target-feature -Xclang -packed-fp32-ops).
"""
import os
import subprocess
import sys
import sysconfig
import tempfile
import warnings
from concurrent.futures import ThreadPoolExecutor
from importlib.machinery import EXTENSION_SUFFIXES
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
SRC = [PKG / "csrc" / "qws_sample.hip", PKG / "csrc" / "qws_verify.hip", PKG / "csrc" / "qws_state.hip", PKG / "csrc" / "qws_pld.hip", PKG / "csrc" / "qws_head.hip",
       PKG / "csrc" / "qws_hooks.hip"]
OUT = PKG / "lib" / "libqws.so"
HOST_SRC, HOST_OUT = PKG / "csrc" / "qws_hostpack.cpp", PKG / "lib" / ("_qws_hostpack" + EXTENSION_SUFFIXES[0])
CXX = os.environ.get("CXX", "g++")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", f"-I{ROOT / 'include'}"]


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    errs = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"compiler failed ({r.returncode}): {' '.join(map(str, cmd))}\n{errs}")


def build(verbose: bool = False) -> Path:
    OUT.parent.mkdir(parents=True, exist_ok=True)
    with tempfile.TemporaryDirectory(prefix="qws_build_") as td:
        objs = [Path(td) / (s.stem + ".o") for s in SRC]
        cmds = [[HIPCC, *FLAGS, "-c", str(s), "-o", str(o)] for s, o in zip(SRC, objs)]
        if verbose:
            for c in cmds:
                print(" ".join(c), flush=True)
        with ThreadPoolExecutor(max_workers=min(len(cmds), os.cpu_count() or 1)) as ex:
            list(ex.map(_run, cmds))
        tmp = OUT.with_suffix(".so.tmp")
        _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)])
        os.replace(tmp, OUT)
    build_host()
    return OUT


def build_host():
    tmp = HOST_OUT.with_suffix(".so.tmp")
    try:
        _run([CXX, "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{sysconfig.get_paths()['include']}", str(HOST_SRC), "-o", str(tmp)])
        os.replace(tmp, HOST_OUT)
    except (RuntimeError, OSError) as e:
        HOST_OUT.unlink(missing_ok=True)  # no older module stays behind
        warnings.warn(f"the host packing module was not built, id lists are packed in Python: {e}", RuntimeWarning)


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))

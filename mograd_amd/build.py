"""Builds libmograd_hip.so (gfx950) from mograd_amd/csrc/*.hip with hipcc, and the host extension
_graph from mograd_amd/native/graph.cpp with g++.

Usage: python -m mograd_amd.build [--force] [--jobs N]

Objects go to mograd_amd/csrc/build/, the library to mograd_amd/libmograd_hip.so.  A
source is recompiled when it or any header is newer than its object.
"""
from __future__ import annotations

import argparse
import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
OBJ_DIR = CSRC / "build"
LIB_PATH = PKG / "libmograd_hip.so"
NATIVE_SRC = PKG / "native" / "graph.cpp"
# Named for the interpreter it is compiled for (_graph.cpython-310-x86_64-linux-gnu.so): another Python
# does not find it and asks for a build instead of loading it.
NATIVE_PATH = PKG / f"_graph{sysconfig.get_config_var('EXT_SUFFIX')}"

ARCH = "gfx950"
# -packed-fp32-ops is switched off: v_pk_*_f32 forms are not to be generated.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]
# -z nodelete: a host that dlopens and later unloads the library must not unmap code that
# late destructors may still run (the hazard the reference's pin.c guards against,
# mograd/runtime/gpu/kernels/pin.c:14-21).
LINK_FLAGS = ["-shared", "-fPIC", f"--offload-arch={ARCH}", "-fno-gpu-rdc", "-Wl,-z,nodelete", "-Wl,--no-undefined"]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found; set HIPCC or install ROCm")


def _headers_mtime() -> float:
    hdrs = list(CSRC.glob("*.h")) + list((ROOT / "include").glob("*.h"))
    return max(h.stat().st_mtime for h in hdrs)


def _compile(hipcc: str, src: Path, obj: Path) -> tuple[Path, int, str]:
    cmd = [hipcc, *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature: harmless.
    noise = ("is not a recognized feature for this target", "packed-fp32-ops")
    err = "\n".join(l for l in proc.stderr.splitlines() if not any(n in l for n in noise))
    return src, proc.returncode, err


def build_native(force: bool = False, verbose: bool = True) -> Path:
    """The CPython extension mograd_amd._graph (host code only)."""
    (PKG / "_graph.so").unlink(missing_ok=True)  # the name it once had, which any Python would load
    newest = max(f.stat().st_mtime for f in (NATIVE_SRC, ROOT / "include" / "mograd_hip.h"))
    if force or not NATIVE_PATH.exists() or NATIVE_PATH.stat().st_mtime < newest:
        cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden",
               f"-I{sysconfig.get_paths()['include']}", f"-I{ROOT / 'include'}", str(NATIVE_SRC), "-o", str(NATIVE_PATH), "-ldl"]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"{NATIVE_SRC.name} failed:\n{proc.stderr}")
        if verbose:
            print(f"[mograd_amd.build] linked {NATIVE_PATH}", flush=True)
    return NATIVE_PATH


def build(force: bool = False, jobs: int | None = None, verbose: bool = True) -> Path:
    build_native(force, verbose)
    hipcc = _hipcc()
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no sources under {CSRC}")
    hdr_time = _headers_mtime()
    todo = []
    objs = []
    for src in sources:
        obj = OBJ_DIR / (src.stem + ".o")
        objs.append(obj)
        if force or not obj.exists() or obj.stat().st_mtime < max(src.stat().st_mtime, hdr_time):
            todo.append((src, obj))
    jobs = jobs or min(8, os.cpu_count() or 1)
    if verbose and todo:
        print(f"[mograd_amd.build] compiling {len(todo)} file(s) for {ARCH} with {jobs} job(s)", flush=True)
    failed = []
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        for src, rc, err in pool.map(lambda so: _compile(hipcc, *so), todo):
            if err.strip() and verbose:
                print(f"--- {src.name}\n{err}", file=sys.stderr, flush=True)
            if rc != 0:
                failed.append(src.name)
    if failed:
        raise RuntimeError(f"hipcc failed for: {', '.join(failed)}")
    if todo or force or not LIB_PATH.exists():
        cmd = [hipcc, *LINK_FLAGS, *map(str, objs), "-o", str(LIB_PATH)]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed:\n{proc.stderr}")
        if verbose:
            print(f"[mograd_amd.build] linked {LIB_PATH}", flush=True)
    return LIB_PATH


def main() -> None:
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--force", action="store_true", help="recompile everything")
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args()
    build(force=args.force, jobs=args.jobs)


if __name__ == "__main__":
    main()

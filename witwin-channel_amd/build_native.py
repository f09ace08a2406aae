"""Build libwcmi.so (all sources under csrc/, HIP ones for gfx950) and
libwcmi_host.so (the plain C++ ones) with ROCm's compilers.

Output: witwin/channel/_native/*.so (in-tree, loaded by
witwin.channel._native). Each source compiles to an object in parallel, then
one link step each produces the shared libraries. The host library lets scene
compilation run before, or without, the GPU runtime.
"""

from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
OUT_DIR = ROOT / "witwin" / "channel" / "_native"
LIB = OUT_DIR / "libwcmi.so"
HOST_LIB = OUT_DIR / "libwcmi_host.so"
BUILD = ROOT / "_build"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HOST_CXX = os.environ.get("HOST_CXX", "/opt/rocm/bin/amdclang++")
ARCH = "gfx950"
# Packed-FP32 instructions are disabled for every kernel: ordinary float code is
# compiled to scalar VALU ops only.
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
HOST_FLAGS = ["-O3", "-std=c++17", "-fPIC"]


def _compile(src: Path) -> Path:
    obj = BUILD / (src.stem + ".o")
    compiler = [HOST_CXX, *HOST_FLAGS] if src.suffix == ".cpp" else [HIPCC, *FLAGS]
    cmd = [*compiler, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compiling {src.name} failed:\n{proc.stderr}")
    return obj


def _link(command: list[str], objects: list[Path], lib: Path) -> None:
    tmp = lib.with_suffix(".so.tmp")
    proc = subprocess.run([*command, "-shared", "-fPIC", *map(str, objects), "-o", str(tmp)], capture_output=True,
                          text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"linking {lib.name} failed:\n{proc.stderr}")
    os.replace(tmp, lib)


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    OUT_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted([*CSRC.glob("*.hip"), *CSRC.glob("*.cpp")])
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(sources))) as pool:
        objects = list(pool.map(_compile, sources))
    _link([HIPCC, f"--offload-arch={ARCH}"], objects, LIB)
    _link([HOST_CXX], [o for o, s in zip(objects, sources) if s.suffix == ".cpp"], HOST_LIB)
    if verbose:
        print(f"built {LIB} and {HOST_LIB.name}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)

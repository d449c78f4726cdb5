"""Builds the HIP kernels into ``dice_amd/libdice_moe.so`` for gfx950.

``python -m dice_amd.build`` (or ``build_library()``) cross-compiles without a
GPU.  Objects go to ``dice_amd/_build/``; the shared library stays in-tree next
to this file so it travels with the source tree.

Every object of the library names the digest of the sources and flags that it was
compiled from (csrc/built_from.h); ``lib.load()`` refuses a library of which any
object's differs from that of the sources beside it.
"""
from __future__ import annotations

import glob
import hashlib
import os
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(HERE, "..", "include")
BUILD_DIR = os.path.join(HERE, "_build")
LIB_PATH = os.path.join(HERE, "libdice_moe.so")

SOURCES = [
    "status.hip",
    "gate.hip",
    "dispatch.hip",
    "combine.hip",
    "modulate.hip",
    "quant.hip",
    "grouped_gemm_f32.hip",
    "grouped_gemm_split.hip",
    "grouped_gemm_bf16.hip",
    "grouped_gemm_f16.hip",
    "grouped_gemm_stream.hip",
    "grouped_gemm_stream_f16.hip",
    "grouped_gemm_persist.hip",
    "grouped_gemm_persist_f16.hip",
    "grouped_gemm_persist_f8.hip",
    "grouped_mlp.hip",
]

# Packed-fp32 VALU forms are switched off for every device translation unit.
HIP_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def source_digest(csrc: str = CSRC, include: str = INCLUDE):
    """Digest of everything a build reads: kernels, headers, generators and flags.  None where the sources are not
    there to build from (a copy of the package without them)."""
    paths = sorted(p for pat in ("*.hip", "*.h", "*.py") for p in glob.glob(os.path.join(csrc, pat)))
    headers = sorted(glob.glob(os.path.join(include, "*.h")))
    if not paths or not headers:
        return None
    h = hashlib.sha256("\0".join(HIP_FLAGS + SOURCES).encode())
    for path in paths + headers:
        with open(path, "rb") as f:
            data = f.read()
        h.update(f"\0{os.path.basename(path)}\0{len(data)}\0".encode())
        h.update(data)
    return h.hexdigest()


_BUILT_FROM = re.compile(rb"dice_moe unit (\S+) ([0-9a-f]{64})\0")


def stale_units(library: bytes, digest: str):
    """The sources whose object in a library (its bytes) is missing or was compiled from anything but `digest`."""
    found = {}
    for m in _BUILT_FROM.finditer(library):
        found.setdefault(m.group(1).decode(), set()).add(m.group(2).decode())
    return [s for s in SOURCES if found.get(s) != {digest}]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the HIP library cannot be built")
    return exe


# Translation units whose kernels keep their sums in accumulation registers that
# the compiler does not know about: their device assembly is kept and checked
# (check_acc_regs.py) before the library is linked.
ACC_CHECKED = {"grouped_gemm_persist.hip", "grouped_gemm_persist_f16.hip", "grouped_gemm_persist_f8.hip"}


def _generate_sources() -> None:
    """Writes the generated k-loops of the expert GEMMs (csrc/gen_persist*_asm.py) into the
    build directory, which is on the include path of every translation unit."""
    import importlib.util
    for name in ("persist64_asm", "persist_dma_asm"):
        spec = importlib.util.spec_from_file_location("gen_" + name, os.path.join(CSRC, f"gen_{name}.py"))
        gen = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(gen)
        text = gen.generate()
        path = os.path.join(BUILD_DIR, name + ".inc")
        if not os.path.exists(path) or open(path).read() != text:
            with open(path, "w") as f:
                f.write(text)


def _remove(path: str) -> None:
    if os.path.exists(path):
        os.remove(path)


def _compile(src: str, extra, digest: str) -> str:
    stem = os.path.splitext(src)[0]
    obj = os.path.join(BUILD_DIR, stem + ".o")
    _remove(obj)                  # (a source that no longer compiles leaves no object of an older one behind)
    cmd = [_hipcc(), *HIP_FLAGS, "-I", BUILD_DIR, f'-DDICE_BUILT_FROM="dice_moe unit {src} {digest}"',
           "-include", os.path.join(CSRC, "built_from.h"), *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    if src in ACC_CHECKED:
        cmd.insert(-4, "-save-temps=obj")
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    if src in ACC_CHECKED:
        from dice_amd.check_acc_regs import check
        try:
            check(os.path.join(BUILD_DIR, stem + "-hip-amdgcn-amd-amdhsa-gfx950.s"))
        except RuntimeError:
            _remove(obj)
            raise
    return obj


def build_library(verbose: bool = True, extra_flags=(), out: str = None) -> str:
    """Compiles every source and links the library (to ``out`` instead of the
    package's own path when given: a second build to compare with, e.g.
    ``python -m dice_amd.build --out /tmp/other.so -DDICE_MFMA_ROWS_OUTERMOST=1``)."""
    target = os.path.abspath(out) if out else LIB_PATH
    _remove(target)               # (a build that fails leaves no library, rather than the one before)
    os.makedirs(BUILD_DIR, exist_ok=True)
    digest = source_digest()      # (before the compiler reads anything: a source edited meanwhile makes its object stale)
    _generate_sources()
    jobs = min(len(SOURCES), max(1, min(8, os.cpu_count() or 1)))
    with ThreadPoolExecutor(jobs) as pool:
        objs = list(pool.map(lambda s: _compile(s, list(extra_flags), digest), SOURCES))
    tmp = target + ".tmp"
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, target)
    if verbose:
        print(f"built {target} ({os.path.getsize(target)} bytes)")
    return target


if __name__ == "__main__":
    argv = sys.argv[1:]
    out_path = None
    if "--out" in argv:
        at = argv.index("--out")
        out_path = argv[at + 1]
        del argv[at:at + 2]
    build_library(extra_flags=argv, out=out_path)

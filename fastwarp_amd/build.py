"""Builds the gfx950 shared library `fastwarp_amd/lib/libfastwarp_hip.so` in-tree with hipcc.

Every translation unit is compiled in parallel into `fastwarp_amd/_build/`, then linked (the CC
kernels as one object per window radius and launch). HIP code is compiled with the packed-FP32 instructions disabled (`-packed-fp32-ops`).
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB = HERE / "lib" / "libfastwarp_hip.so"
BUILD = HERE / "_build"

SOURCES = [
    CSRC / "hip" / "kernels.hip",
    CSRC / "hip" / "mi_kernels.hip",
    CSRC / "hip" / "backend.hip",
    CSRC / "hip" / "mi_backend.hip",
    CSRC / "hip" / "noalloc.hip",
    CSRC / "hip" / "batch.hip",
    CSRC / "capi.cpp",
    CSRC / "serve.cpp",
]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FW_OFFLOAD_ARCH", "gfx950")
FLAGS = [
    "-std=c++17",
    "-O3",
    f"--offload-arch={ARCH}",
    "-fPIC",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wno-unused-result",
    f"-I{HERE.parent / 'include'}",
]


def _run(cmds: list[list[str]]) -> None:
    def one(c):
        p = subprocess.run(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        return p.returncode, p.stdout

    # as many at a time as there are processors (a large CC object takes about 0.5 GB)
    with ThreadPoolExecutor(max_workers=os.cpu_count() or 1) as pool:
        done = list(pool.map(one, cmds))
    failed = []
    for c, (code, out) in zip(cmds, done):
        if code != 0:
            lines = [l for l in out.splitlines() if "packed-fp32-ops" not in l and "unknown target feature" not in l]
            failed.append((c, "\n".join(lines)))
    if failed:
        for c, text in failed:
            sys.stderr.write(" ".join(c) + "\n" + text + "\n")
        raise RuntimeError(f"{len(failed)} compile step(s) failed")


def objects() -> list[tuple[Path, Path, list[str]]]:
    """(source, object, further flags) of every compile step, the longest ones first."""
    cc = CSRC / "hip" / "cc.hip"
    steps = [(cc, BUILD / f"cc_r{r}_{part}.o", [f"-DFW_CC_RADIUS={r}", f"-DFW_CC_PART={part}"])
             for r in range(8, 0, -1) for part in (1, 0, 2)]
    return steps + [(src, BUILD / (src.name + ".o"), []) for src in SOURCES]


def build(verbose: bool = False) -> Path:
    BUILD.mkdir(exist_ok=True)
    LIB.parent.mkdir(exist_ok=True)
    steps = objects()
    _run([[HIPCC, *FLAGS, *extra, "-c", str(src), "-o", str(obj)] for src, obj, extra in steps])
    tmp = LIB.with_suffix(".so.tmp")
    _run([[HIPCC, *FLAGS, "-shared", *[str(obj) for _, obj, _ in steps], "-o", str(tmp), "-lpthread"]])
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)

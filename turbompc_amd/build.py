"""Builds libtmpc_hip.so for gfx950 in-tree (turbompc_amd/lib/).

Two translation units, compiled side by side: csrc/resident.hip (the on-chip ADMM
path) and csrc/capi.hip (every other kernel and the C ABI).  All HIP code is
compiled with packed-FP32 instructions disabled.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from pathlib import Path

PKG = Path(__file__).resolve().parent
SOURCES = [PKG / "csrc" / n for n in ("capi.hip", "resident.hip")]
OUT = PKG / "lib" / "libtmpc_hip.so"
ARCH = os.environ.get("TMPC_OFFLOAD_ARCH", "gfx950")


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise FileNotFoundError("hipcc not found (set HIPCC or install ROCm)")


def build_library(verbose: bool = False) -> Path:
    OUT.parent.mkdir(parents=True, exist_ok=True)
    flags = [f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
    with tempfile.TemporaryDirectory(prefix="build_", dir=OUT.parent) as tmp:
        objs = [Path(tmp) / (src.stem + ".o") for src in SOURCES]
        cmds = [[hipcc(), *flags, "-c", str(src), "-o", str(obj)] for src, obj in zip(SOURCES, objs)]
        procs = [subprocess.Popen(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for c in cmds]
        logs = [p.communicate()[0] for p in procs]
        new = Path(tmp) / OUT.name
        link = [hipcc(), f"--offload-arch={ARCH}", "-fPIC", "-shared", "-o", str(new), *map(str, objs)]
        for p, c, log in zip(procs, cmds, logs):
            if p.returncode != 0:
                sys.stderr.write(log)
                raise RuntimeError(f"hipcc failed ({p.returncode}): {' '.join(c)}")
        r = subprocess.run(link, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError(f"hipcc failed ({r.returncode}): {' '.join(link)}")
        if verbose:
            sys.stderr.write("".join(logs) + r.stderr)
        os.replace(new, OUT)
    return OUT


if __name__ == "__main__":
    print(build_library(verbose=True))

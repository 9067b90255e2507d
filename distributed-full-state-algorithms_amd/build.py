"""Build libfsa.so (HIP kernels + C ABI) for gfx950 with hipcc.

    python distributed-full-state-algorithms_amd/build.py [-j JOBS] [--verbose]

Objects go to distributed-full-state-algorithms_amd/_build/, the library to
distributed-full-state-algorithms_amd/libfsa.so (in-tree, so it travels with
the repository snapshot).  Every HIP translation unit is compiled with packed
FP32 instructions disabled.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OUT_DIR = PKG / "_build"
LIB = PKG / "libfsa.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FSA_OFFLOAD_ARCH", "gfx950")

COMMON = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-command-line-argument",
    f"-I{PKG.parent / 'include'}",
]

# Kernels that interpret op lists with uniform branches over a large register
# state: structurizing those branches (the default, needed only for divergent
# ones) copies the state at every merge.  With it the reverse register-tile
# kernels spill 248 (FP64) and 510 (FP32) VGPRs, without it none.  The file's
# other kernels have the same registers or fewer (k_pauli_groups 98 against 128).
UNIFORM = ["-mllvm", "-structurizecfg-skip-uniform-regions"]
PER_FILE = {"kernels_reduce.hip": UNIFORM}


def sources():
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")))


def _compile(src: Path, verbose: bool) -> Path:
    obj = OUT_DIR / (src.stem + src.suffix.replace(".", "_") + ".o")
    lang = ["-x", "hip"] if src.suffix == ".hip" else []
    cmd = [HIPCC, *COMMON, *PER_FILE.get(src.name, []), *lang, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{r.stdout}\n{r.stderr}")
    warn = "\n".join(l for l in r.stderr.splitlines()
                     if "packed-fp32-ops" not in l and l.strip() and "warning: feature" not in l)
    if warn and verbose:
        print(warn, file=sys.stderr)
    return obj


def build(jobs: int = 8, verbose: bool = False) -> Path:
    OUT_DIR.mkdir(exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose), srcs))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=8)
    ap.add_argument("--verbose", action="store_true")
    a = ap.parse_args()
    print(build(a.j, a.verbose))

"""Builds the braidinfer_amd C-ABI shared library for gfx950 with hipcc.

Usage:  python -m braidinfer_amd.build [--jobs N]

Every ``csrc/*.hip`` file is compiled to an object in parallel, then linked
into ``braidinfer_amd/lib/libbraidinfer_amd.so``.  The library is the product:
the Python package loads it and fails loudly when it is missing.  The package's
own calls go through ``lib/_bfa_entry.<ABI tag>.so`` (csrc/pyentry.cpp), built for
the interpreter that builds; without that interpreter's headers, or under another
interpreter, they go through ctypes, 1 to 5 us a call slower.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
INCLUDE = ROOT / "include"
LIBDIR = PKG / "lib"
OBJDIR = LIBDIR / "obj"
LIBNAME = "libbraidinfer_amd.so"
ENTRYNAME = "_bfa_entry" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so")
ARCH = "gfx950"

# -ffp-contract=off keeps every product and sum separately rounded, the way the
# reference's unfused torch op chains compute them.  -packed-fp32-ops is
# disabled so no v_pk_{add,mul,fma}_f32 is emitted.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build braidinfer_amd")
    return exe


def _compile(src: Path) -> Path:
    obj = OBJDIR / (src.stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{proc.stdout}\n{proc.stderr}")
    return obj


def _build_entry() -> Path | None:
    """The CPython module over the library (csrc/pyentry.cpp), next to it; None where
    this interpreter's headers are not installed."""
    headers = Path(sysconfig.get_paths()["include"])
    if not (headers / "Python.h").exists():
        print(f"{ENTRYNAME} not built: no Python.h in {headers}; calls go through ctypes")
        return None
    tmp = LIBDIR / (ENTRYNAME + ".tmp")
    cmd = [hipcc(), "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-Wall", f"-I{INCLUDE}", f"-I{headers}",
           str(CSRC / "pyentry.cpp"), "-shared", f"-L{LIBDIR}", f"-l:{LIBNAME}", "-Wl,-rpath,$ORIGIN", "-o", str(tmp)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"building {ENTRYNAME} failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, LIBDIR / ENTRYNAME)
    return LIBDIR / ENTRYNAME


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    """Compiles every csrc/*.hip file and links the shared library; returns its path."""
    OBJDIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = jobs or min(len(sources), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, sources))
    out = LIBDIR / LIBNAME
    tmp = LIBDIR / (LIBNAME + ".tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, out)
    _build_entry()
    if verbose:
        print(f"built {out}")
    return out


def main(argv=None) -> int:
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--jobs", type=int, default=None)
    args = ap.parse_args(argv)
    build(args.jobs, verbose=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())

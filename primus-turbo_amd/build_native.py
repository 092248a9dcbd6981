"""Build libprimus_turbo_amd.so (the C-ABI library) with hipcc for gfx950, and libprimus_turbo_torch-<torch's version>.so
(the host side of the dense torch operators, csrc/torch_ops.cpp) with the host compiler against the installed torch. Without
torch the C library is all that there is to build.

Usage:  python primus-turbo_amd/build_native.py [--force] [-j N]

Every ``csrc/*.hip`` translation unit is compiled to an object file under
``primus-turbo_amd/build/`` and linked into ``primus-turbo_amd/lib/``. hipcc
cross-compiles for gfx950, so no GPU is needed to build.
"""

from __future__ import annotations

import argparse
import importlib.util
import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import check_asm

ROOT = Path(__file__).resolve().parent
CSRC = ROOT / "csrc"
BUILD = ROOT / "build"
LIBDIR = ROOT / "lib"
LIBNAME = "libprimus_turbo_amd.so"
HEADER = ROOT.parent / "include" / "primus_turbo_amd.h"

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-fno-gpu-rdc",
    # hipcc -O3 may otherwise form packed-fp32 VALU ops from scalar float code
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wno-unused-result",
]


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (looked at $HIPCC, PATH and /opt/rocm/bin)")


def lib_path() -> Path:
    return LIBDIR / LIBNAME


def torch_lib_path() -> Path | None:
    """The library for the installed torch (its C++ interface is that version's alone), None without one."""
    if importlib.util.find_spec("torch") is None:
        return None
    import torch

    return LIBDIR / f"libprimus_turbo_torch-{torch.__version__}.so"


def _build_torch_ops(force: bool, verbose: bool) -> Path | None:
    """One host translation unit on torch's headers; the HIP runtime is the one that torch ships."""
    src, out = CSRC / "torch_ops.cpp", torch_lib_path()
    if out is None:
        return None
    if not force and out.exists() and out.stat().st_mtime >= max(src.stat().st_mtime, HEADER.stat().st_mtime):
        return out
    import torch

    root = Path(torch.__file__).resolve().parent
    rocm = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-isystem", str(root / "include"), "-isystem", str(rocm / "include"), str(src), "-o", str(out),
           f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-lamdhip64", "-ldl"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{src.name} failed:\n{res.stderr}")
    return out


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _deps_mtime() -> float:
    deps = list(CSRC.glob("*.h")) + [HEADER]
    return max(p.stat().st_mtime for p in deps)


def _extra_flags(src: Path) -> list[str]:
    """Per-file compiler flags: a leading ``// hipcc-flags: ...`` comment line in the source."""
    with open(src) as f:
        first = f.readline()
    tag = "// hipcc-flags:"
    return first[len(tag):].split() if first.startswith(tag) else []


def _compile_one(hipcc: str, src: Path, force: bool, verbose: bool) -> Path:
    obj = BUILD / (src.stem + ".o")
    if not force and obj.exists():
        if obj.stat().st_mtime >= max(src.stat().st_mtime, _deps_mtime()):
            return obj
    with tempfile.TemporaryDirectory(dir=BUILD) as tmp:  # (for the assembly, which is looked at before the object counts)
        made = Path(tmp) / obj.name
        cmd = [hipcc, *HIPCC_FLAGS, *_extra_flags(src), "-save-temps=obj", "-c", str(src), "-o", str(made)]
        if verbose:
            print(" ".join(cmd), flush=True)
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode == 0:
            asm = Path(tmp) / f"{src.stem}-hip-amdgcn-amd-amdhsa-{ARCH}.s"
            check_asm.check(asm.read_text().split("\n"), src.name)
            made.replace(obj)
    # the host pass warns that it does not know the packed-fp32 feature: harmless
    err = "\n".join(
        l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip()
    )
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err and verbose:
        print(err, file=sys.stderr)
    return obj


def build(force: bool = False, jobs: int | None = None, verbose: bool = False) -> Path:
    hipcc = hipcc_path()
    BUILD.mkdir(exist_ok=True)
    LIBDIR.mkdir(exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no .hip sources under {CSRC}")
    jobs = jobs or min(8, len(srcs))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        torch_ops = ex.submit(_build_torch_ops, force, verbose)
        objs = list(ex.map(lambda s: _compile_one(hipcc, s, force, verbose), srcs))
    out = lib_path()
    cmd = [hipcc, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", str(out)] + [str(o) for o in objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    torch_ops.result()  # (a failure there leaves the C library built)
    return out


def ensure_built() -> Path:
    """Return the library path, building the libraries only when one does not exist yet."""
    out, torch_out = lib_path(), torch_lib_path()
    if not out.exists() or (torch_out is not None and not torch_out.exists()):
        build()
    return out


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("-j", type=int, default=None)
    ap.add_argument("-q", "--quiet", action="store_true")
    a = ap.parse_args()
    p = build(force=a.force, jobs=a.j, verbose=not a.quiet)
    print(f"built {p}")

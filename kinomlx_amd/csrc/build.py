"""Build ``kinomlx_amd/libkx355.so`` from ``csrc/*.hip`` with hipcc for gfx950, and
``kinomlx_amd/_host.so``, the native launch path over it, from ``csrc/host.cpp`` with g++.

Run as ``python -m kinomlx_amd.csrc.build`` (or through ``__graft_entry__.build()``). Objects go
to ``_build/`` at the repository root; the shared libraries are written next to the package so that
they travel with the source tree.
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

CSRC = Path(__file__).resolve().parent
PACKAGE = CSRC.parent
ROOT = PACKAGE.parent
INCLUDE = ROOT / "include"
BUILD = ROOT / "_build"
LIBRARY = PACKAGE / "libkx355.so"
HOST_MODULE = PACKAGE / "_host.so"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    f"-I{INCLUDE}",
    # No packed-fp32 VALU instructions (v_pk_*_f32) anywhere.
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
]


def _hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(found).exists():
        raise RuntimeError("hipcc not found: the kx355 HIP library cannot be built")
    return found


def _compile(source: Path) -> Path:
    obj = BUILD / (source.stem + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-c", str(source), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {source.name}:\n{proc.stderr}")
    return obj


def _compile_host() -> None:
    """The CPython module of ``host.cpp``: torch's headers and libraries, no HIP code."""
    import torch
    from torch.utils import cpp_extension

    tmp = HOST_MODULE.with_suffix(".so.tmp")
    includes = [str(INCLUDE), sysconfig.get_paths()["include"], *cpp_extension.include_paths()]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{p}" for p in includes),
           str(CSRC / "host.cpp"), "-o", str(tmp), *(f"-L{p}" for p in cpp_extension.library_paths()),
           "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{proc.stderr}")
    os.replace(tmp, HOST_MODULE)


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    """Compile every ``csrc/*.hip``, link ``libkx355.so`` and build ``_host.so``; returns the library path."""
    BUILD.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError("no HIP sources found")
    workers = jobs or min(len(sources) + 1, max(1, min(8, os.cpu_count() or 1)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=workers) as pool:
        host = pool.submit(_compile_host)
        objects = list(pool.map(_compile, sources))
        host.result()
    tmp = LIBRARY.with_suffix(".so.tmp")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-o", str(tmp), *map(str, objects)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"linking libkx355.so failed:\n{proc.stderr}")
    os.replace(tmp, LIBRARY)
    if verbose:
        print(f"built {LIBRARY} from {len(sources)} sources", file=sys.stderr)
    return LIBRARY


if __name__ == "__main__":
    build(verbose=True)

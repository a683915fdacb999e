"""Builds libpto_hip.so (HIP kernels + C ABI) for gfx950 and the Python extension beside it, in-tree.

    python -m pypto_amd.build [--force]

Every ``csrc/*.hip`` is compiled with hipcc for ``--offload-arch=gfx950`` and linked into
``pypto_amd/lib/libpto_hip.so``, which needs neither torch nor Python; hipcc cross-compiles without a GPU present.
``pyext/dispatch.cpp`` is host code for torch's Python binding and becomes ``pypto_amd/lib/_dispatch.<Python
ABI>.torch-<version>.so`` afterwards, where torch is installed.
"""

from __future__ import annotations

import argparse
import importlib.util
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

from ._lib import dispatch_path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIB_DIR = PKG / "lib"
OBJ_DIR = LIB_DIR / "obj"
LIB_PATH = LIB_DIR / "libpto_hip.so"
INCLUDE = PKG.parent / "include"
DISPATCH_SRC = PKG / "pyext" / "dispatch.cpp"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-fno-gpu-rdc",
    # keep the compiler from forming packed fp32 ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]


# Per-file additions.  The attention kernels keep their MFMA accumulators in architectural VGPRs
# (they are rescaled by VALU code every chunk); the GEMM keeps the default AGPR form.
EXTRA_FLAGS = {
    "paged_attention.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _stale(target: Path, deps: list[Path]) -> bool:
    if not target.exists():
        return True
    t = target.stat().st_mtime
    return any(d.stat().st_mtime > t for d in deps)


def _compile(src: Path, force: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    headers = list(CSRC.glob("*.h")) + list(INCLUDE.glob("*.h"))
    if force or _stale(obj, [src] + headers):
        cmd = [HIPCC, *FLAGS, *EXTRA_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src.name}:\n{r.stderr}")
        err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
        if err.strip():
            sys.stderr.write(err + "\n")
    return obj


def _build_dispatch(force: bool) -> None:
    import torch

    # named after the Python and the torch it is compiled for: another one's binary is never taken for up to date
    target = dispatch_path()
    if not force and not _stale(target, [DISPATCH_SRC, *INCLUDE.glob("*.h")]):
        return
    root = Path(torch.__file__).resolve().parent
    cmd = [CXX, "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", f"-I{INCLUDE}",
           f"-I{sysconfig.get_paths()['include']}", f"-I{root / 'include'}", f"-I{root / 'include/torch/csrc/api/include'}",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", str(DISPATCH_SRC), "-o", str(target),
           f"-L{root / 'lib'}", "-ltorch_python", "-ltorch_cpu", "-lc10"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{CXX} failed for {DISPATCH_SRC.name}:\n{r.stderr}")


def build(force: bool = False, jobs: int | None = None) -> Path:
    """Compile and link; returns the path of the shared library."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(8, len(srcs))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
    if force or _stale(LIB_PATH, objs):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB_PATH), *map(str, objs)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stderr}")
    if importlib.util.find_spec("torch") is None:
        sys.stderr.write(f"torch is not installed: {DISPATCH_SRC.name} is left out\n")
    else:
        _build_dispatch(force)
    return LIB_PATH


def main() -> None:
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--force", action="store_true", help="recompile everything")
    args = ap.parse_args()
    print(build(force=args.force))


if __name__ == "__main__":
    main()

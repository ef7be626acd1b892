"""Build libm5k.so (gfx950 HIP kernels + C ABI) in-tree with hipcc.

Every translation unit under ``csrc/`` is compiled to an object under ``_build/``
(in parallel), then linked into ``lib/libm5k.so`` next to this package.  The measurement
kernels under ``diag/`` (bench.py's MFMA ceiling) go into ``lib/libm5k_diag.so``, the native
front of the linears and projections under ``binding/`` (host code, against torch's headers) into
``lib/m5k_fast.so``; where those headers are missing the other two are built all the same.
Flags:

* ``--offload-arch=gfx950`` only: MI355X is the single target.
* ``-ffp-contract=off``: no FMA contraction, so FP32 epilogues and normalization keep
  the rounding sequence the contract spells out.
* ``-fhip-fp32-correctly-rounded-divide-sqrt``: IEEE ``/`` and ``sqrt`` (the
  quantizer's ``x / scale`` must round exactly like the CPU reference).
* ``-Xclang -target-feature -Xclang -packed-fp32-ops``: no packed FP32 VALU ops.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import warnings
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_ROOT = Path(__file__).resolve().parent.parent  # m5-max-kernels_amd/
REPO_ROOT = PKG_ROOT.parent
CSRC = PKG_ROOT / "csrc"
INCLUDE = REPO_ROOT / "include"
BUILD_DIR = REPO_ROOT / "_build" / "libm5k"
LIB_PATH = PKG_ROOT / "lib" / "libm5k.so"
DIAG_DIR = PKG_ROOT / "diag"
DIAG_LIB_PATH = PKG_ROOT / "lib" / "libm5k_diag.so"
FAST_SRC = PKG_ROOT / "binding" / "fast_ops.cpp"
FAST_PATH = PKG_ROOT / "lib" / "m5k_fast.so"

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build libm5k.so")
    return path


def sources() -> list[Path]:
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")))


def _compile(src: Path, force: bool) -> Path:
    obj = BUILD_DIR / (src.name + ".o")
    headers = list(CSRC.glob("*.h")) + list(INCLUDE.glob("*.h"))
    newest_dep = max(p.stat().st_mtime for p in [src, *headers])
    if not force and obj.exists() and obj.stat().st_mtime >= newest_dep:
        return obj
    cmd = [hipcc(), *HIPCC_FLAGS, f"-I{INCLUDE}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd = [hipcc(), "-O2", "-std=c++17", "-fPIC", f"-I{INCLUDE}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{proc.stderr[-4000:]}")
    return obj


def build(force: bool = True, jobs: int | None = None, verbose: bool = False) -> Path:
    """Compile every csrc/ translation unit for gfx950 and link lib/libm5k.so."""
    BUILD_DIR.mkdir(parents=True, exist_ok=True)
    LIB_PATH.parent.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        fast = pool.submit(_compile_fast, force)
        objs = list(pool.map(lambda s: _compile(s, force), srcs))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link of libm5k.so failed:\n{proc.stderr[-4000:]}")
    os.replace(tmp, LIB_PATH)
    build_diag()
    # The library stands by itself; the front is built beside it, and an older one does not stay there.
    FAST_PATH.unlink(missing_ok=True)
    if (fast_obj := fast.result()) is not None:
        _link_fast(fast_obj)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources, and {DIAG_LIB_PATH}", file=sys.stderr)
    return LIB_PATH


def _front_includes() -> list[str]:
    """Include folders of the native front, or none where g++, Python's or torch's headers are not
    installed: libm5k.so needs none of them."""
    try:
        from torch.utils.cpp_extension import include_paths
    except ImportError:  # setuptools, which torch's extension builder imports
        return []
    python, folders = sysconfig.get_paths()["include"], include_paths()
    if not (shutil.which("g++") and (Path(python) / "Python.h").exists()
            and any((Path(p) / "torch" / "extension.h").exists() for p in folders)):
        return []
    return [f"-I{python}", *(f"-isystem{p}" for p in folders)]


def _compile_fast(force: bool) -> Path | None:
    """The native front of the linears and projections: host code against torch's headers (None without
    them: the checks then run in Python)."""
    import torch

    includes = _front_includes()
    if not includes:
        warnings.warn("g++, Python.h or torch's headers are missing: m5k_fast.so is not built", RuntimeWarning)
        return None
    obj = BUILD_DIR / f"fast_ops-{torch.__version__}.o"  # an object of another torch is no object of this one
    newest_dep = max(p.stat().st_mtime for p in [FAST_SRC, *INCLUDE.glob("*.h")])
    if not force and obj.exists() and obj.stat().st_mtime >= newest_dep:
        return obj
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DM5K_TORCH_VERSION="{torch.__version__}"', f"-I{INCLUDE}", *includes, "-c", str(FAST_SRC), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile of {FAST_SRC.name} failed:\n{proc.stderr[-4000:]}")
    return obj


def _link_fast(obj: Path) -> None:
    from torch.utils.cpp_extension import library_paths

    tmp = FAST_PATH.with_suffix(".so.tmp")
    cmd = ["g++", "-shared", "-o", str(tmp), str(obj), f"-L{LIB_PATH.parent}", "-lm5k", "-Wl,-rpath,$ORIGIN",
           *(f"-L{p}" for p in library_paths()), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link of {FAST_PATH.name} failed:\n{proc.stderr[-4000:]}")
    os.replace(tmp, FAST_PATH)


def build_diag() -> Path:
    """Link lib/libm5k_diag.so: measurement kernels used by bench.py (no op uses them)."""
    tmp = DIAG_LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), *HIPCC_FLAGS, "-shared", "-o", str(tmp), *map(str, sorted(DIAG_DIR.glob("*.hip")))]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"build of libm5k_diag.so failed:\n{proc.stderr[-4000:]}")
    os.replace(tmp, DIAG_LIB_PATH)
    return DIAG_LIB_PATH


if __name__ == "__main__":
    build(force="--incremental" not in sys.argv, verbose=True)

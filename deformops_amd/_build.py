"""Ahead-of-time build of the HIP library for gfx950 and of its native torch bridge.

libdeformops_amd.so is the MSDA library (the C ABI of include/deformops_amd.h),
built in-tree (``deformops_amd/lib/``) with hipcc and loaded with ctypes; _native.so is
the Python extension module that plain eager calls go through (csrc/bridge.cpp, host
code only). Nothing is compiled at import or call time.

    python -m deformops_amd._build
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from pathlib import Path

__all__ = ["ARCH", "HIPCC_FLAGS", "LIBRARY", "SOURCES", "build", "compile_library"]

PACKAGE_DIR = Path(__file__).resolve().parent
REPO_DIR = PACKAGE_DIR.parent
SOURCES = [PACKAGE_DIR / "csrc" / "msda.hip"]
INCLUDE_DIR = REPO_DIR / "include"
LIBRARY = PACKAGE_DIR / "lib" / "libdeformops_amd.so"
BRIDGE_SOURCE = PACKAGE_DIR / "csrc" / "bridge.cpp"
BRIDGE = PACKAGE_DIR / "lib" / "_native.so"
ARCH = os.environ.get("DEFORMOPS_AMD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++20",
    "-fPIC",
    "-shared",
    # Packed fp32 VALU ops stay off: hipcc forms them from ordinary float code.
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    f"-I{INCLUDE_DIR}",
]


def _hipcc() -> str:
    for candidate in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if candidate and Path(candidate).exists():
            return candidate
    msg = "hipcc not found; set HIPCC or install ROCm"
    raise FileNotFoundError(msg)


def build(*, verbose: bool = False) -> Path:
    """Compile the MSDA library, atomically replacing it; return its path.

    Raises
    ------
    subprocess.CalledProcessError
        If hipcc fails; the compiler output is in the exception.
    """
    build_bridge(verbose=verbose)
    return compile_library(SOURCES, LIBRARY, verbose=verbose)


def build_bridge(*, verbose: bool = False) -> Path:
    """Compile the native torch bridge (host code), atomically replacing it."""
    import torch  # noqa: PLC0415
    from torch.utils import cpp_extension  # noqa: PLC0415

    rocm = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "include"
    includes = [*cpp_extension.include_paths(), str(rocm), sysconfig.get_paths()["include"]]
    command = [
        os.environ.get("CXX") or shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared",
        "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",  # noqa: SLF001
        f"-I{INCLUDE_DIR}", *(f"-isystem{path}" for path in dict.fromkeys(includes)), str(BRIDGE_SOURCE),
        *(f"-L{path}" for path in cpp_extension.library_paths()),
        "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python",
    ]
    return _compile(command, BRIDGE, verbose=verbose)


def compile_library(sources: list[Path], target: Path, *, verbose: bool) -> Path:
    return _compile([_hipcc(), *HIPCC_FLAGS, *map(str, sources)], target, verbose=verbose)


def _compile(command: list[str], target: Path, *, verbose: bool) -> Path:
    """Run ``command -o target``, through a temporary directory beside it: the linker
    makes the file itself, so that its mode follows the umask (a file made for it by
    ``mkstemp`` keeps 0600, and only its owner could load the library)."""
    target.parent.mkdir(parents=True, exist_ok=True)
    with tempfile.TemporaryDirectory(prefix=target.name + ".", suffix=".tmp", dir=target.parent) as folder:
        built = Path(folder) / target.name
        cmd = [*command, "-o", str(built)]
        result = subprocess.run(cmd, capture_output=True, text=True, check=False)  # noqa: S603
        if verbose or result.returncode != 0:
            noise = "is not a recognized feature for this target"
            lines = [ln for ln in (result.stdout + result.stderr).splitlines() if noise not in ln]
            if lines:
                print("\n".join(lines), file=sys.stderr)
        if result.returncode != 0:
            raise subprocess.CalledProcessError(result.returncode, cmd, result.stdout, result.stderr)
        os.replace(built, target)
    return target


if __name__ == "__main__":
    print(build(verbose=True))

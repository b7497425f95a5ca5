"""Build the gfx950 C-ABI library ``my_vllm_amd/lib/libmy_vllm_amd.so``.

Every ``csrc/*.hip`` translation unit is compiled with ``hipcc`` for gfx950
only and linked into one shared library that exports the ``extern "C"`` entry
points declared in ``include/my_vllm_amd.h``; ``csrc/host_ops.cpp`` becomes
``lib/mva_host.so``, the Python operators' launch path over it.  The library is built in-tree so
that it travels with the source tree; no JIT cache is involved.

Run ``python -m my_vllm_amd.build`` (or ``__graft_entry__.build()``).
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
CSRC_DIR = PACKAGE_DIR / "csrc"
LIB_DIR = PACKAGE_DIR / "lib"
LIB_PATH = LIB_DIR / "libmy_vllm_amd.so"
HOST_PATH = LIB_DIR / "mva_host.so"
BUILD_DIR = PACKAGE_DIR / "_build"

OFFLOAD_ARCH = "gfx950"
# Packed fp32 VALU forms are disabled for every kernel of this library.  The
# atomic optimizer is off: it turns a single-lane atomic into a wave-wide
# reduction whose result is broadcast right after the atomic, which makes the
# decode kernel's piece claims wait for every load in flight.
HIP_FLAGS = (
    f"--offload-arch={OFFLOAD_ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-mllvm",
    "-amdgpu-atomic-optimizer-strategy=None",
)


def _hipcc() -> str:
    candidates = (
        os.environ.get("HIPCC"),
        "/opt/rocm/bin/hipcc",
        shutil.which("hipcc"),
    )
    for candidate in candidates:
        if candidate and Path(candidate).exists():
            return candidate
    raise RuntimeError("hipcc not found; the gfx950 library cannot be built")


def _compile(hipcc: str, source: Path, obj: Path) -> None:
    cmd = [hipcc, *HIP_FLAGS, f"-I{CSRC_DIR}", "-c", str(source), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(
            f"hipcc failed for {source.name}:\n{proc.stdout}\n{proc.stderr}"
        )


def _build_host_module(target: Path) -> None:
    """Compile ``csrc/host_ops.cpp`` (host code only) against torch's headers
    into ``target``, bound to the library beside it."""
    import torch

    from . import _native

    root = Path(torch.__file__).resolve().parent
    cmd = [
        os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++") or "g++",
        "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
        "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-DMVA_HOST_ABI_VERSION={_native.ABI_VERSION}",
        f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        f"-I{root / 'include'}", "-I/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}",
        str(CSRC_DIR / "host_ops.cpp"), "-o", str(target),
        f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-lamdhip64", "-ltorch_cpu", "-ltorch_python",
        f"-L{target.parent}", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN",
    ]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for host_ops.cpp:\n{proc.stdout}\n{proc.stderr}")


def build(verbose: bool = False) -> Path:
    """Compile all kernels for gfx950 and link the shared library; return its path.

    The library and the host module over it are put in place together, once
    both are built: a build that fails leaves the earlier pair.  They are
    written by the compilers themselves, so that their modes follow the umask
    and another user's processes can load them."""
    hipcc = _hipcc()
    sources = sorted(CSRC_DIR.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC_DIR}")
    BUILD_DIR.mkdir(exist_ok=True)
    LIB_DIR.mkdir(exist_ok=True)
    objects = [BUILD_DIR / (src.stem + ".o") for src in sources]
    jobs = max(1, min(len(sources), int(os.environ.get("MAX_JOBS", "8"))))
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(lambda pair: _compile(hipcc, *pair), zip(sources, objects)))
    with tempfile.TemporaryDirectory(prefix=".build.", dir=LIB_DIR) as tmp:
        library, host = Path(tmp) / LIB_PATH.name, Path(tmp) / HOST_PATH.name
        cmd = [hipcc, f"--offload-arch={OFFLOAD_ARCH}", "-shared", "-fPIC", "-o", str(library), *map(str, objects)]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
        _build_host_module(host)
        os.replace(library, LIB_PATH)
        os.replace(host, HOST_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(sources)} sources", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)

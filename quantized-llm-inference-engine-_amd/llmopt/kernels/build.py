"""Build ``libllmopt_qlinear.so`` from ``csrc/*.hip`` with hipcc for gfx950, and the torch binding of
the linears' host path, ``_llmopt_torch.so``, from ``csrc/torch_binding.cpp`` with g++.

Usage: ``python -m llmopt.kernels.build`` (or :func:`build_library`). Objects go to
``<package>/_build/``; the library is written next to this file so it ships with the
source tree. The library's run path lists torch's bundled ROCm libraries first, so the
process uses one HIP runtime whichever of torch and this library is loaded first.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
PACKAGE_ROOT = HERE.parent.parent  # quantized-llm-inference-engine-_amd/
CSRC = PACKAGE_ROOT / "csrc"
INCLUDE = PACKAGE_ROOT.parent / "include"
BUILD_DIR = PACKAGE_ROOT / "_build"
LIBRARY = HERE / "libllmopt_qlinear.so"
BINDING = HERE / "_llmopt_torch.so"  # the linears' host path (csrc/torch_binding.cpp)
ARCH = os.environ.get("LLMOPT_OFFLOAD_ARCH", "gfx950")

COMPILE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    # The dequantization must round exactly like the reference's torch code: no
    # contraction of (q - z) * s into an fma, and fp32 denormals kept.
    "-ffp-contract=off",
    "-fno-gpu-flush-denormals-to-zero",
    # Packed fp32 arithmetic stays off on this target.
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def _hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(found).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build the kernels")
    return found


def _torch_lib_dir() -> str | None:
    try:
        import torch
    except ImportError:  # pragma: no cover - torch is a hard dependency of the package
        return None
    return str(Path(torch.__file__).resolve().parent / "lib")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def build_library(verbose: bool = False, jobs: int | None = None) -> Path:
    """Compile every ``csrc/*.hip`` and link the shared library. Always rebuilds."""
    hipcc = _hipcc()
    BUILD_DIR.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")

    def compile_one(src: Path) -> Path:
        obj = BUILD_DIR / (src.stem + ".o")
        cmd = [hipcc, *COMPILE_FLAGS, f"-I{INCLUDE}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src.name}:\n{proc.stdout}\n{proc.stderr}")
        return obj

    workers = jobs or min(len(srcs), 8)
    with ThreadPoolExecutor(max_workers=workers) as pool:
        binding = pool.submit(build_binding_if_possible, verbose)
        objs = list(pool.map(compile_one, srcs))
        binding.result()

    tmp = LIBRARY.with_suffix(".so.tmp")
    link = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    torch_lib = _torch_lib_dir()
    if torch_lib:
        link.append(f"-Wl,-rpath,{torch_lib}")
    # hipBLASLt for the two-pass prefill's dense GEMM.
    link += ["-L/opt/rocm/lib", "-lhipblaslt"]
    if verbose:
        print(" ".join(link), flush=True)
    proc = subprocess.run(link, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, LIBRARY)
    return LIBRARY


def build_binding(verbose: bool = False) -> Path:
    """Compile ``csrc/torch_binding.cpp`` against torch into ``_llmopt_torch.so``. Always rebuilds."""
    import sysconfig

    import torch

    root = Path(torch.__file__).resolve().parent
    src, tmp = CSRC / "torch_binding.cpp", BINDING.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "c++", "-O2", "-fPIC", "-shared", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-isystem{root / 'include'}", f"-isystem{root / 'include/torch/csrc/api/include'}",
           f"-isystem{sysconfig.get_paths()['include']}", f"-isystem{_rocm_include()}", str(src), "-o", str(tmp),
           f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python",
           f"-Wl,-rpath,{root / 'lib'}"]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed on {src.name}:\n{proc.stdout}\n{proc.stderr}")
    os.replace(tmp, BINDING)
    return BINDING


def build_binding_if_possible(verbose: bool = False) -> Path | None:
    """:func:`build_binding`, or None (and no binding left from an earlier build) where it does not
    compile: the kernel library needs neither torch's headers nor a host compiler of its own, and
    works without it."""
    try:
        return build_binding(verbose)
    except (ImportError, OSError, RuntimeError) as exc:
        BINDING.unlink(missing_ok=True)
        print(f"the linears' native host path is left out: {exc}", file=sys.stderr, flush=True)
        return None


def _rocm_include() -> str:
    return str(Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "include")


def main() -> int:
    path = build_library(verbose="-v" in sys.argv)
    print(path)
    return 0


if __name__ == "__main__":
    raise SystemExit(main())

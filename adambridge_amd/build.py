"""Build libadambridge_hip.so (gfx950) in-tree with hipcc.

    python -m adambridge_amd.build

Flags: -O3; -ffp-contract=off (products and sums round separately except where
the source writes an FMA, as the reference's kernels do); HIP's default
correctly rounded FP32 division and sqrt and kept denormals (no fast-math);
packed FP32 instructions disabled for device code.
"""

from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
import tempfile
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
SOURCES = [PKG / "csrc" / name for name in ("adambridge_hip.hip", "abh_state.hip", "abh_loss.hip", "abh_gemm.hip")]
LIB = PKG / "libadambridge_hip.so"
BIND_SOURCE = PKG / "csrc" / "abh_bind.cpp"   # host code over torch's C++ tensors: the Python module _bind
BIND = PKG / "_bind.so"
ARCH = os.environ.get("ADAMBRIDGE_HIP_ARCH", "gfx950")


def hipcc() -> str:
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cand = Path(rocm) / "bin" / "hipcc"
    return str(cand) if cand.exists() else "hipcc"


def flags() -> list[str]:
    return [f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
            "-ffp-contract=off", "-fno-fast-math", "-fvisibility=hidden",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wall", "-Wno-unused-result",
            f"-I{ROOT / 'include'}"]


def bind_command(out: Path) -> list[str]:
    import torch
    from torch.utils import cpp_extension

    lib = Path(torch.__file__).resolve().parent / "lib"
    includes = [f"-I{d}" for d in (ROOT / "include", *cpp_extension.include_paths(), sysconfig.get_paths()["include"])]
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes, str(BIND_SOURCE),
            "-o", str(out), f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-lc10"]


def build(verbose: bool = False) -> Path:
    """Compile the library and the host module (always; a stale one is never reused): the sources side by
    side, then one link."""
    with tempfile.TemporaryDirectory(prefix="adambridge_build_") as work:
        objects = [Path(work) / (src.stem + ".o") for src in SOURCES]
        compiles = [[hipcc(), *flags(), "-c", str(src), "-o", str(obj)] for src, obj in zip(SOURCES, objects)]
        tmp, bind = LIB.with_suffix(".so.tmp"), BIND.with_suffix(".so.tmp")
        compiles.append(bind_command(bind))
        link = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objects), "-o", str(tmp)]
        if verbose:
            print("\n".join(" ".join(cmd) for cmd in [*compiles, link]), file=sys.stderr)
        running = [subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
                   for cmd in compiles]
        results = [(proc.communicate()[0], proc.returncode) for proc in running]
        linked = None
        if all(code == 0 for _, code in results):
            linked = subprocess.run(link, capture_output=True, text=True)
            results.append((linked.stderr, linked.returncode))
        for output, code in results:
            if code != 0:
                raise RuntimeError(f"the compiler failed ({code}):\n{output}")
        os.replace(tmp, LIB)
        os.replace(bind, BIND)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))

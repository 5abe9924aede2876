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
import tempfile
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
SOURCES = [PKG / "csrc" / name for name in ("adambridge_hip.hip", "abh_state.hip", "abh_loss.hip")]
LIB = PKG / "libadambridge_hip.so"
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


def build(verbose: bool = False) -> Path:
    """Compile the library (always; a stale library is never reused): the sources side by side, then
    one link."""
    with tempfile.TemporaryDirectory(prefix="adambridge_build_") as work:
        objects = [Path(work) / (src.stem + ".o") for src in SOURCES]
        compiles = [[hipcc(), *flags(), "-c", str(src), "-o", str(obj)] for src, obj in zip(SOURCES, objects)]
        tmp = LIB.with_suffix(".so.tmp")
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
                raise RuntimeError(f"hipcc failed ({code}):\n{output}")
        os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))

"""Build recipe of the gfx950 kernel library ``libqepw_hip.so`` (in-tree).

``python -m qe_python_amd.build`` compiles every ``csrc/*.hip`` with hipcc
for gfx950 and links them into ``qe_python_amd/libqepw_hip.so``, the C-ABI
library declared in ``include/qepw.h``.  Packed-FP32 instructions are
disabled for all device code (``-Xclang -target-feature -Xclang
-packed-fp32-ops``).
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
OBJ = ROOT / "_build" / "obj"
LIB = PKG / "libqepw_hip.so"
ARCH = os.environ.get("QEPW_OFFLOAD_ARCH", "gfx950")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result", "-I", str(ROOT / "include"),
]


# per-file flags: the FFT kernels feed literal zeros into their register DFTs
# for the grid slots outside the sphere, and x + 0 folds to x only when the
# sign of zero may be ignored
EXTRA_FLAGS = {"qepw_fft.hip": ["-fno-signed-zeros"],
               # contraction off: the grouped and one-problem plane kernels agree
               # bit for bit (their fused multiply-adds are written out)
               "qepw_plane_c128.hip": ["-fno-signed-zeros", "-ffp-contract=off"],
               "qepw_plane_c64.hip": ["-fno-signed-zeros", "-ffp-contract=off"]}


def _compile(src: Path) -> Path:
    obj = OBJ / (src.stem + ".o")
    cmd = [HIPCC, *FLAGS, *EXTRA_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr[-6000:]}")
    return obj


def build(verbose: bool = False) -> Path:
    OBJ.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp),
           *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr[-6000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)

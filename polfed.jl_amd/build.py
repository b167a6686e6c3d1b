"""In-tree build of libpolfed_hip.so for gfx950 with hipcc.

The shared library is written next to the package (``lib/libpolfed_hip.so``)
so that it travels with the source tree; nothing is installed elsewhere.
"""
from __future__ import annotations

import concurrent.futures
import os
import pathlib
import subprocess
import tempfile

PKG = pathlib.Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OUT = PKG / "lib" / "libpolfed_hip.so"
SOURCES = ["ops.hip", "team.hip", "qteam.hip", "batch.hip", "packed.hip", "dense.hip", "capi.cpp"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed FP32 instructions are kept out of every kernel of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _run(cmd, verbose: bool) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    if verbose or res.returncode != 0:
        msg = "\n".join(l for l in (res.stdout + res.stderr).splitlines()
                        if "packed-fp32-ops" not in l)
        if msg.strip():
            print(msg)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}): {' '.join(cmd)}")


def build_library(verbose: bool = False) -> pathlib.Path:
    """Compile every HIP source into lib/libpolfed_hip.so (always rebuilds)."""
    OUT.parent.mkdir(parents=True, exist_ok=True)
    tmp = OUT.with_suffix(".so.tmp")
    with tempfile.TemporaryDirectory() as d:  # the sources compile side by side
        objs = [str(pathlib.Path(d) / (s + ".o")) for s in SOURCES]
        cmds = [[HIPCC, *FLAGS, "-c", "-o", o, str(CSRC / s)] for s, o in zip(SOURCES, objs)]
        with concurrent.futures.ThreadPoolExecutor(os.cpu_count() or 1) as pool:
            list(pool.map(lambda c: _run(c, verbose), cmds))
        _run([HIPCC, *FLAGS, "-shared", "-o", str(tmp), *objs], verbose)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build_library(verbose=True))

"""Builds libytm.so (the HIP kernels + C-ABI) for gfx950, in-tree next to this file.

    python -m ytm_amd.build_lib
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
CSRC = HERE / "csrc"
SOURCES = [CSRC / "ytm_kernels.hip", CSRC / "ytm_api.hip", CSRC / "ytm_jit.hip", CSRC / "ytm_binarize.hip",
           CSRC / "ytm_matrix.hip", CSRC / "ytm_memory.hip"]
OUT = HERE / "libytm.so"
# Device headers that the run-time specialised compile (hipRTC) needs, embedded as text.
JIT_HEADERS = ["ytm_types.h", "ytm_device.h", "ytm_train.h"]
JIT_INC = CSRC / "gen_jit_sources.inc"

HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "--offload-arch=gfx950",
    # exact IEEE semantics for the parity-critical float/double compares and updates
    "-ffp-contract=off",
    # packed-fp32 VALU forms off
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{ROOT / 'include'}",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found")


def write_jit_sources() -> None:
    """Writes gen_jit_sources.inc: the device headers as raw string literals."""
    delim = "ytmsrc"
    parts = ["// Generated by ytm_amd/build_lib.py from " + ", ".join(JIT_HEADERS) + ". Do not edit.\n"]
    for h in JIT_HEADERS:
        text = (CSRC / h).read_text()
        if f'){delim}"' in text:
            raise RuntimeError(f"{h} contains the raw-string delimiter")
        parts.append(f'static const char kJitSrc_{h.replace(".", "_")}[] = R"{delim}({text}){delim}";\n')
    parts.append("static const char* const kJitHeaderSources[] = {"
                 + ", ".join(f'kJitSrc_{h.replace(".", "_")}' for h in JIT_HEADERS) + "};\n")
    parts.append("static const char* const kJitHeaderNames[] = {" + ", ".join(f'"{h}"' for h in JIT_HEADERS) + "};\n")
    parts.append(f"static const int kJitHeaderCount = {len(JIT_HEADERS)};\n")
    text = "".join(parts)
    if not JIT_INC.exists() or JIT_INC.read_text() != text:
        JIT_INC.write_text(text)


def build(verbose: bool = False) -> Path:
    write_jit_sources()
    tmp = OUT.with_suffix(".so.tmp")
    cmd = [hipcc(), *HIPCC_FLAGS, "-o", str(tmp), *map(str, SOURCES), "-lhiprtc"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{res.stdout}\n{res.stderr}")
    if verbose and res.stderr:
        print(res.stderr, file=sys.stderr)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))

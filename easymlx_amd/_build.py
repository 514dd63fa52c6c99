"""In-tree build of ``easymlx_amd/_lib/libemx_attn.so`` with hipcc for gfx950."""

from __future__ import annotations

import os
import shutil
import subprocess

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
SOURCES = [os.path.join(CSRC, f) for f in ("emx_attn.hip", "emx_mfma.hip")]
DEPENDS = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hpp", ".hip"))]
OUT = os.path.join(_HERE, "_lib", "libemx_attn.so")

HIPCC_FLAGS = [
    "-O3",
    "--offload-arch=gfx950",
    "-std=c++17",
    "-fPIC",
    # no packed-fp32 VALU ops anywhere in device code
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    # leading kernel arguments arrive in SGPRs with the wave (gfx950 kernel-argument preload)
    "-mllvm",
    "-amdgpu-kernarg-preload-count=16",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found (ROCm required to build libemx_attn.so)")
    return path


def build_native(verbose: bool = False) -> str:
    """Compile the HIP library; always recompiles.  Returns the .so path."""
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    tmp = OUT + ".tmp"
    objs = [os.path.join(os.path.dirname(OUT), os.path.basename(src) + ".o") for src in SOURCES]
    cmds = [[hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj] for src, obj in zip(SOURCES, objs)]
    # one compiler per translation unit, side by side
    procs = [subprocess.Popen(c, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True) for c in cmds]
    errs = [p.communicate()[1] for p in procs]
    link = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    for cmd, p, err in zip(cmds, procs, errs):
        if p.returncode != 0:
            raise RuntimeError(f"hipcc failed ({p.returncode}):\n{' '.join(cmd)}\n{err[-4000:]}")
    res = subprocess.run(link, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{' '.join(link)}\n{res.stderr[-4000:]}")
    if verbose:
        print("\n".join(" ".join(c) for c in [*cmds, link]))
    os.replace(tmp, OUT)
    return OUT

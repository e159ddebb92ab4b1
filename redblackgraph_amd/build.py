"""Build recipe for librbg_hip.so (gfx950).

Run as ``python -m redblackgraph_amd.build``.  Compiles every ``csrc/*.hip``
file into one shared library next to this file.  hipcc cross-compiles for
gfx950 without a GPU present.
"""
from __future__ import annotations

import glob
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "librbg_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed FP32 instructions stay disabled in every device build
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result", "-Wno-unused-command-line-argument",
]


_SHIFT = re.compile(r"^\s*v_(?:lshlrev_b64|lshrrev_b64|ashrrev_i64)\S*\s+v\[\d+:\d+\],\s*v(\d+),")


def shift_hazards(asm: str):
    """Kernels of a gfx950 assembly text with a 64-bit shift whose amount lies
    in the last VGPR the wave is allocated (blocks of eight): the hardware then
    reads a register that is not the wave's (the last-register bug LLVM works
    round on gfx90a), and the result changes from run to run."""
    found, name, amounts, vgprs = [], None, [], 0
    for line in asm.splitlines():
        m = re.match(r"^(_Z\w+):", line)
        if m:
            name, amounts = m.group(1), []
            continue
        m = _SHIFT.match(line)
        if m:
            amounts.append(int(m.group(1)))
            continue
        m = re.match(r"\s*\.amdhsa_accum_offset (\d+)", line)  # the VGPRs allocated below the accumulators
        if m:
            vgprs = int(m.group(1))
        elif re.match(r"\s*\.end_amdhsa_kernel", line) and name:
            if (vgprs - 1) in amounts and vgprs % 8 == 0:
                found.append(name)
            name = None
    return found


def _asm_paths(src: str, objdir: str):
    stem = os.path.splitext(os.path.basename(src))[0]
    return glob.glob(os.path.join(objdir, f"{stem}-hip-amdgcn-*gfx950*.s"))


def _check_asm(src: str, objdir: str) -> None:
    paths = _asm_paths(src, objdir)
    if not paths:
        raise RuntimeError(f"{src}: no device assembly to check in {objdir}")
    for path in paths:
        with open(path) as f:
            bad = shift_hazards(f.read())
        if bad:
            raise RuntimeError(f"{src}: 64-bit shift by the last allocated VGPR in {', '.join(bad)}")


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def build(verbose: bool = False, jobs: int = 8) -> str:
    """Compile each source to an object in parallel, then link."""
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    procs = []
    objs = []
    for src in sources():
        obj = os.path.join(objdir, os.path.basename(src) + ".o")
        objs.append(obj)
        for old in _asm_paths(src, objdir):  # the check reads this build's
            os.remove(old)
        cmd = [HIPCC, *FLAGS, "--save-temps=obj", "-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        if len(procs) >= jobs:
            _drain(procs)
    _drain(procs)
    for src in sources():
        _check_asm(src, objdir)
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


def _drain(procs):
    while procs:
        cmd, p = procs.pop(0)
        out, _ = p.communicate()
        if p.returncode != 0:
            sys.stderr.write(out.decode(errors="replace"))
            raise RuntimeError(f"hipcc failed: {' '.join(cmd)}")
        elif out:
            txt = out.decode(errors="replace")
            # hipcc's host pass warns about the device-only target feature
            lines = [ln for ln in txt.splitlines() if "packed-fp32-ops" not in ln and ln.strip()]
            if lines:
                sys.stderr.write("\n".join(lines) + "\n")


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))

"""Build libhqekv.so (hand-written HIP for gfx950) and _host.so (the host side of the calls, C++ over torch) in-tree.

``python -m hqekv_amd.build`` compiles every source under ``hqekv_amd/csrc`` and links
``hqekv_amd/libhqekv.so`` with hipcc, which cross-compiles for gfx950 without a GPU, and ``hqekv_amd/_host.so`` with the
host compiler.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
LIB = PKG / "libhqekv.so"
HOST = PKG / "_host.so"
SOURCES = ["capi.hip", "quant_pack.hip", "attn.hip", "decode_qk.hip", "decode_pv.hip", "decode_step.hip", "decode_static.hip", "migrate.hip", "reconstruct.hip", "planner.hip", "importance.hip", "prompt_attn.hip"]

HIPCC_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
    # packed-FP32 VALU forms are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # a kernel's first 14 argument words arrive in scalar registers
    "-mllvm", "-amdgpu-kernarg-preload-count=14",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
    f"-I{ROOT / 'include'}", f"-I{CSRC}",
]


# A workgroup of decode_step.hip that has waited long enough loops over whole tiles; what the compiler would move out of that
# loop it keeps on the stack.
EXTRA_FLAGS = {"decode_step.hip": ["-mllvm", "-disable-machine-licm"]}


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "is not a recognized feature" not in l)
    if r.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(map(str, cmd)) + "\n" + out)
    return out


def _build_host(objdir: Path) -> str:
    """_host.so: torch's headers and libraries, no device code."""
    import torch
    base, rocm = Path(torch.__file__).resolve().parent, Path(_hipcc()).resolve().parents[1]
    tmp = objdir / "_host.so.tmp"
    log = _run([os.environ.get("CXX") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                f"-I{ROOT / 'include'}", f"-I{base / 'include'}", f"-I{base / 'include/torch/csrc/api/include'}", f"-I{rocm / 'include'}",
                "-I/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}", str(CSRC / "host.cpp"), "-o", str(tmp), f"-L{base / 'lib'}",
                "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ltorch_hip", "-ldl"])
    os.replace(tmp, HOST)
    return log


def build(verbose: bool = False) -> Path:
    hipcc = _hipcc()
    objdir = PKG / "build"
    objdir.mkdir(exist_ok=True)
    objs = [objdir / (Path(s).stem + ".o") for s in SOURCES]

    def compile_one(pair):
        src, obj = pair
        return _run([hipcc, *HIPCC_FLAGS, *EXTRA_FLAGS.get(src, []), "-c", str(CSRC / src), "-o", str(obj)])

    with ThreadPoolExecutor(max_workers=min(4, len(SOURCES))) as ex:
        host = ex.submit(_build_host, objdir)
        logs = list(ex.map(compile_one, zip(SOURCES, objs)))
        logs.append(host.result())
    tmp = LIB.with_suffix(".so.tmp")
    logs.append(_run([hipcc, "-shared", "-fPIC", "--offload-arch=gfx950", *map(str, objs), "-o", str(tmp)]))
    os.replace(tmp, LIB)
    if verbose:
        for l in logs:
            if l.strip():
                print(l)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
    sys.exit(0)

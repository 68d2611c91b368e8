"""Build libmt_attn.so, libmt_torch.so (and the bench-only libmt_probe.so) in-tree.

Run as ``python mega-trading_amd/build_lib.py`` or through
``__graft_entry__.build()``.  The libraries land next to this file so they
travel with the source tree (they are git-ignored, not installed anywhere).

* libmt_attn.so: the gfx950 kernels and their C ABI (hipcc).
* libmt_torch.so: the PyTorch-ROCm side of the ops -- the GPU
  implementations and the autograd of the ``mega_trading_amd::*`` ops whose
  schemas and shapes ``attention.py``, ``ops.py`` and ``projection.py`` declare
  -- built with the host compiler against torch's headers and linked to
  libmt_attn.so; no device code.
* libmt_probe.so: a sustained-MFMA-rate probe that bench.py reports beside
  the roofline; it is not part of the attention ABI.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_NAME = "libmt_attn.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
SOURCES = ["mt_attention.hip", "mt_ops.hip"]
PROBE_NAME = "libmt_probe.so"
PROBE_PATH = os.path.join(HERE, PROBE_NAME)
PROBE_SOURCES = ["mfma_probe.hip"]
HEADERS = ["mt_common.h", "attn_kernels.h", "lds_tile.h", "mt_abi.h", "ops_kernels.h"]
ARCH = "gfx950"


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build libmt_attn.so")
    return path


def compile_command(out: str = LIB_PATH, sources: list[str] | None = None) -> list[str]:
    return [
        hipcc(),
        f"--offload-arch={ARCH}",
        "-O3",
        "-std=c++17",
        "-fPIC",
        "-shared",
        # never let the compiler form packed-fp32 ALU ops (v_pk_{add,mul,fma}_f32)
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wno-pass-failed",
        # one soname for every build, so the attention ops library binds to
        # whichever libmt_attn.so the process loaded first
        "-Wl,-soname," + os.path.basename(LIB_PATH if sources is None else out).replace(".tmp", ""),
        "-o", out,
        *[os.path.join(CSRC, s) for s in (SOURCES if sources is None else sources)],
    ]


TORCH_OPS_NAME = "libmt_torch.so"
TORCH_OPS_PATH = os.path.join(HERE, TORCH_OPS_NAME)
TORCH_OPS_SOURCES = ["mt_torch.cpp"]


def torch_ops_command(out: str = TORCH_OPS_PATH) -> list[str]:
    import torch

    tdir = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    return [
        shutil.which("g++") or "g++",
        "-O2", "-std=c++17", "-fPIC", "-shared",
        f"-D_GLIBCXX_USE_CXX11_ABI={abi}", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        "-I", os.path.join(tdir, "include"),
        "-I", os.path.join(tdir, "include", "torch", "csrc", "api", "include"),
        "-I", os.path.join(rocm, "include"),
        *[os.path.join(CSRC, s) for s in TORCH_OPS_SOURCES],
        "-L", os.path.join(tdir, "lib"), "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip",
        "-L", HERE, "-l:" + LIB_NAME,
        "-Wl,-rpath,$ORIGIN", "-Wl,-rpath," + os.path.join(tdir, "lib"),
        "-o", out,
    ]


def build(verbose: bool = False) -> str:
    """Compile every library (always; a stale build is never reused)."""
    _compile(PROBE_PATH, PROBE_SOURCES, verbose)
    path = _compile(LIB_PATH, SOURCES, verbose)
    _run(TORCH_OPS_PATH, torch_ops_command(TORCH_OPS_PATH + ".tmp"), verbose)
    return path


def _run(path: str, cmd: list[str], verbose: bool) -> str:
    tmp = path + ".tmp"
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({proc.returncode}):\n{proc.stderr}")
    os.replace(tmp, path)
    return path


def _compile(path: str, sources: list[str], verbose: bool) -> str:
    tmp = path + ".tmp"
    cmd = compile_command(tmp, sources)
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)
    os.replace(tmp, path)
    return path


if __name__ == "__main__":
    print(build(verbose=True))

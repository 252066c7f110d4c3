"""Build recipe for libmega_hip.so (hand-written HIP kernels for gfx950 + the C ABI).

Run as a script (`python fairseq-apollo_amd/build.py`) or through
`__graft_entry__.build()`.  hipcc cross-compiles for gfx950 without a GPU.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmega_hip.so")
HOST = os.path.join(HERE, "mega_host.so")

SOURCES = [
    "gemm16_wide.hip", "gemm16_wide_f16.hip", "attention_wide.hip",      # (the longest first)
    "capi.hip",
    "timestep_norm.hip",
    "timestep_norm_bwd.hip",
    "sequence_norm.hip",
    "ema_scan.hip",
    "ema_mfma.hip",
    "norm_ema_fused.hip",
    "ema_rows.hip",
    "ema_bwd.hip", "ema_bwd_tile.hip",
    "decode.hip",
    "decode_layer.hip",
    "elementwise.hip",
    "gemm.hip", "gemm16.hip",
    "gate_glue.hip",
    "embed_grad.hip",
    "row_norm.hip",
    "attention.hip",
    "attention_mfma.hip",
    "long_conv.hip",
    "param_prep.hip",
]

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-fno-gpu-rdc",
    # packed fp32 instructions are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result", "-Wno-unused-value",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def build_library(verbose: bool = True, jobs: int = 8) -> str:
    """Compile every source to an object in parallel, then link the shared library."""
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    cc = hipcc()
    procs = []
    objs = []
    compile_flags = [f for f in FLAGS if f != "-shared"]
    for src in SOURCES:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        objs.append(obj)
        cmd = [cc, *compile_flags, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        while sum(p.poll() is None for _, p in procs) >= jobs:
            for _, p in procs:
                if p.poll() is None:
                    p.wait()
                    break
    failed = False
    for src, p in procs:
        out, _ = p.communicate()
        if p.returncode != 0:
            failed = True
            sys.stderr.write(f"--- {src} failed ---\n{out}\n")
        elif verbose and out.strip():
            # the host pass warns that it does not know the packed-fp32 feature: harmless
            lines = [l for l in out.splitlines() if "packed-fp32-ops" not in l and l.strip()]
            if lines:
                print("\n".join(lines))
    if failed:
        raise RuntimeError("hipcc failed")
    cmd = [cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    build_host(verbose)
    return LIB


def build_host(verbose: bool = True) -> str:
    """The Python extension of native host code (csrc/host.cpp): C++ against torch's headers, no device code; it
    finds libmega_hip.so beside itself."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    tlib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f"-I{d}" for d in (*include_paths(), sysconfig.get_paths()["include"])], os.path.join(CSRC, "host.cpp"), "-o", HOST,
           f"-L{HERE}", "-l:libmega_hip.so", f"-L{tlib}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return HOST


if __name__ == "__main__":
    build_library()

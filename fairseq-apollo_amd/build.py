"""Build recipe for libmega_hip.so (hand-written HIP kernels for gfx950 + the C ABI).

Run as a script (`python fairseq-apollo_amd/build.py`) or through
`__graft_entry__.build()`.  hipcc cross-compiles for gfx950 without a GPU.
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys
import tempfile

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


def assembly_faults(name: str, listing: list, matrix: bool = True) -> list:
    """What a kernel with inline assembly must not hold, in its disassembly (lines of llvm-objdump).  Loads to LDS: M0 is
    written before one and used for nothing else.  Matrix instructions: the compiler pads those it knows with wait states, these
    it moves values around unpadded.  Two wait states belong between a vector instruction and a matrix instruction that
    shares a register with it, 19 between a matrix instruction and any other use of its result; no registers in scratch memory
    (fragments would come back through copies)."""
    code, at = [], {}
    for line in listing:
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)", line)
        if m:
            at[int(m[3], 16)] = len(code)
            jump = re.search(r"\+0x([0-9a-f]+)>", m[4]) if m[1].startswith(("s_branch", "s_cbranch")) else None
            code.append((m[1], m[2], jump and int(jump[1], 16)))
    start = min(at, default=0)
    before = [[i - 1] if i and code[i - 1][0] not in ("s_branch", "s_endpgm") else [] for i in range(len(code))]
    for i, (_, _, jump) in enumerate(code):
        if jump is not None:
            before[at[start + jump]].append(i)

    def registers(text):
        out = set()
        for kind, low, _, high in re.findall(r"\b([va])\[?(\d+)(:(\d+))?", text):
            out |= {(kind, r) for r in range(int(low), int(high or low) + 1)}
        return out

    uses = [registers(args) for _, args, _ in code]
    results = [registers(args.split(",")[0]) for _, args, _ in code]

    def within(i, states):
        """Instructions from which fewer than `states` wait states lie before i, along every way there."""
        seen, todo = {}, [(j, states) for j in before[i]]
        while todo:
            j, left = todo.pop()
            if seen.get(j, 0) >= left:
                continue
            seen[j] = left
            left -= 1 + (int(code[j][1], 0) if code[j][0] == "s_nop" else 0)
            if left > 0:
                todo += [(k, left) for k in before[j]]
        return seen

    faults = []
    for i, (op, args, _) in enumerate(code):
        if re.search(r"\bm0\b", args) and not (op == "s_mov_b32" and args.startswith("m0,") and
                                               any(code[k][0].startswith("global_load_lds") for k in (i + 1, i + 2) if k < len(code))):
            faults.append(f"{name}: M0 beside the loads to LDS: {op} {args}")
        if not matrix:
            continue
        if op.startswith("v_mfma"):
            for j in within(i, 2):
                if code[j][0].startswith("v_") and not code[j][0].startswith("v_mfma") and uses[j] & uses[i]:
                    faults.append(f"{name}: {code[j][0]} {code[j][1]} just before {op} {args}")
        elif any(kind == "a" for kind, _ in uses[i]):
            for j in within(i, 19):
                if code[j][0].startswith("v_mfma") and results[j] & uses[i]:
                    faults.append(f"{name}: {op} {args} too close behind {code[j][0]} {code[j][1]}")
        if op.startswith("scratch_"):
            faults.append(f"{name}: registers in scratch memory: {op} {args}")
    return faults


# kernels with loads to LDS as assembly (dma16 of gemm16_wide.h), and whether their matrix instructions are assembly too
ASSEMBLY = {"gemm16_square_kernel": True, "gemm16_tall_kernel": False, "attn_wide_kernel": False}


def check_assembly(lib: str) -> dict:
    """assembly_faults of every kernel in a built library that holds assembly; how many there are of each."""
    objdump = os.path.join(os.path.dirname(os.path.realpath(shutil.which(hipcc()) or hipcc())), "..", "llvm", "bin", "llvm-objdump")
    faults, kernels = [], dict.fromkeys(ASSEMBLY, 0)
    with tempfile.TemporaryDirectory() as folder:
        os.symlink(os.path.abspath(lib), os.path.join(folder, "lib"))
        subprocess.check_call([objdump, "--offloading", "lib"], cwd=folder, stdout=subprocess.DEVNULL)
        for part in sorted(os.listdir(folder)):
            path = os.path.join(folder, part)
            if "gfx950" not in part or not any(kind.encode() in open(path, "rb").read() for kind in ASSEMBLY):
                continue
            text = subprocess.check_output([objdump, "-d", "--no-show-raw-insn", path], text=True)
            for block in re.split(r"\n(?=[0-9a-f]+ <)", text):
                head, _, body = block.partition("\n")
                for kind, matrix in ASSEMBLY.items():
                    if kind in head:
                        kernels[kind] += 1
                        faults += assembly_faults(head.split("<")[1].split(">")[0], body.splitlines(), matrix)
    if faults:
        raise RuntimeError("inline assembly in the compiled kernels:\n" + "\n".join(faults[:20]))
    return kernels


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
    check_assembly(LIB)
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

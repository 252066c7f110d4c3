"""The build's check of kernels with inline assembly (no GPU): what it finds in listings with a mistake, and that the built
library holds none."""
import importlib.util
import os

import pytest

from conftest import ROOT

spec = importlib.util.spec_from_file_location("mega_build_recipe", os.path.join(ROOT, "fairseq-apollo_amd", "build.py"))
build = importlib.util.module_from_spec(spec)
spec.loader.exec_module(build)

MFMA = "v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]"


def faults(*code):
    """of instructions of four bytes each; a jump names its target's number in the list"""
    lines = []
    for i, text in enumerate(code):
        op, _, args = text.partition(" ")
        target = ""
        if op.startswith(("s_branch", "s_cbranch")):
            target, args = f" <kernel+0x{4 * int(args):x}>", "1"
        lines.append(f"\t{op} {args}    // {0x100 + 4 * i:012X}: 00000000{target}")
    return build.assembly_faults("kernel", lines)


@pytest.mark.parametrize("count,code", [
    (1, ("v_mov_b32_e32 v5, v20", MFMA)),                                        # a fragment moved just before
    (1, ("v_mov_b32_e32 v5, v20", "s_nop 0", MFMA)),                             # one wait state of two
    (0, ("v_mov_b32_e32 v5, v20", "s_nop 1", MFMA)),
    (0, ("v_mov_b32_e32 v5, v20", "s_add_u32 s0, s0, 4", "ds_read_b128 v[20:23], v30", MFMA)),
    (0, ("v_mov_b32_e32 v12, v20", MFMA)),                                       # another register
    (1, ("v_accvgpr_write_b32 a3, v20", MFMA)),
    (3, (MFMA, "s_nop 7", "v_accvgpr_read_b32 v20, a2", "v_mov_b32_e32 v8, 0", MFMA)),
    (0, (MFMA, "s_nop 15", "s_nop 15", "v_accvgpr_read_b32 v20, a2")),
    (1, (MFMA, "s_nop 1", "global_store_dwordx4 v20, a[0:3], s[0:1]")),
    (0, (MFMA, MFMA, "v_mfma_f32_16x16x32_bf16 a[4:7], v[4:7], v[8:11], a[4:7]")),
    (1, (MFMA, "s_nop 4", "v_mov_b32_e32 v9, v20", "s_cbranch_scc1 0")),         # around a loop
    (0, (MFMA, "s_nop 4", "v_mov_b32_e32 v9, v20", "s_branch 5", "s_nop 0", "s_nop 2", MFMA)),
    (1, ("scratch_load_dwordx4 v[4:7], off, off offset:16", "s_waitcnt vmcnt(0)", MFMA)),
    (0, ("s_mov_b32 m0, s4", "s_nop 0", "global_load_lds_dwordx4 v3, s[0:1]")),
    (1, ("s_mov_b32 m0, s4", "s_nop 0", "v_movrels_b32_e32 v3, v4")),
    (1, ("s_add_u32 s4, m0, 4",)),
])
def test_mistakes_are_found(count, code):
    assert len(faults(*code)) == count


def test_the_built_kernels():
    """both types, every order of the operands (attention: its three products), with and without a partial step"""
    assert build.check_assembly(build.LIB) == {"gemm16_square_kernel": 16, "gemm16_tall_kernel": 16, "attn_wide_kernel": 12}

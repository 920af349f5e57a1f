"""Generated-code check of the kernels whose matrix instructions stand in asm statements (no GPU needed: hipcc cross-compiles to assembly).
See isa_mfma.py for the hazard."""
import os
import re
import shutil
import subprocess

import pytest

from isa_lint import copies_of_inflight_registers
from isa_mfma import asm_matrix_instructions, broken_wait_states

CSRC = os.path.join(os.path.dirname(__file__), "..", "yscv_amd", "csrc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-S", "--cuda-device-only"]
# the sources with asm matrix instructions, and their extra flags in the Makefile
SOURCES = {"int4_gemm_wide.hip": [], "i8_gemm_wide.hip": ["-ffp-contract=off"]}


def _asm(*lines):
    return "\n".join(["_Zkernel:"] + ["\t;;#ASMSTART\n\t%s\n\t;;#ASMEND" % l[1:] if l[0] == "!" else "\t" + l if l[0] != "." else l for l in lines])


MFMA = "!v_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[8:11], a[0:3]"


@pytest.mark.parametrize("lines,hits", [
    # an operand that is written right in front, one instruction in front, two in front; by an asm statement as well
    (["v_mov_b32_e32 v5, 0", MFMA], 1),
    (["v_mov_b32_e32 v5, 0", "s_add_u32 s0, s0, 1", MFMA], 1),
    (["v_mov_b32_e32 v5, 0", "s_nop 1", MFMA], 0),
    (["!v_xor_b32 v8, s0, v8", MFMA], 1),
    (["v_accvgpr_write_b32 a3, 0", MFMA], 1),
    # the result: read, written again, copied for another accumulator, added to in part and added to as a whole
    ([MFMA, "s_nop 6", "v_accvgpr_read_b32 v0, a2"], 1),
    ([MFMA, "s_nop 7", "v_accvgpr_read_b32 v0, a2"], 0),
    ([MFMA, "v_accvgpr_mov_b32 a9, a0"], 1),
    ([MFMA, "v_accvgpr_write_b32 a1, 0"], 1),
    ([MFMA, "!v_mfma_i32_16x16x64_i8 a[2:5], v[4:7], v[8:11], a[2:5]"], 1),
    ([MFMA, MFMA], 0),
    # round a loop, and on one of two ways only
    ([".LBB0_1:", "v_mov_b32_e32 v0, v9", MFMA, "s_nop 7", "v_mov_b32_e32 v8, v0", "s_cbranch_scc1 .LBB0_1", "s_endpgm"], 0),
    ([".LBB0_1:", MFMA, "s_nop 7", "v_mov_b32_e32 v8, v0", "s_cbranch_scc1 .LBB0_1", "s_endpgm"], 1),
    (["s_cbranch_scc1 .LBB0_2", MFMA, ".LBB0_2:", "v_accvgpr_read_b32 v0, a2"], 1),
    (["!v_mfma_f32_32x32x16_f16 a[0:15], v[4:7], v[8:11], a[0:15]"], 1),  # not in the table
])
def test_checker(lines, hits):
    assert len(broken_wait_states(_asm(*lines))) == hits


def test_buffer_loads_to_lds_are_counted():
    asm = "\n".join([
        "_Zkernel:",
        "\t;;#ASMSTART", "\tglobal_load_dwordx4 v[4:7], v1, s[2:3]", "\t;;#ASMEND",
        "\t;;#ASMSTART", "\tbuffer_load_dwordx4 v9, s[4:7], s8 offen lds", "\t;;#ASMEND",
        "\t;;#ASMSTART", "\ts_waitcnt vmcnt(1)", "\t;;#ASMEND",
        "\tv_mov_b32_e32 v12, v6",
        "\ts_endpgm"])
    assert copies_of_inflight_registers(asm) == []  # the load to LDS is the one that is left
    early = asm.replace("vmcnt(1)", "vmcnt(2)")
    assert [h[3] for h in copies_of_inflight_registers(early)] == [3]


def test_every_source_with_asm_matrix_instructions_is_named():
    found = {f for f in os.listdir(CSRC) if f.endswith((".hip", ".hpp")) and re.search(r'asm[^;]*"v_(mfma|smfmac)', open(os.path.join(CSRC, f)).read())}
    assert found == set(SOURCES)


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
@pytest.mark.parametrize("name", sorted(SOURCES))
def test_matrix_instructions_have_their_wait_states(name, tmp_path_factory):
    # (the check of loads in flight compiles the same sources with the same flags, for minutes: what it has left in this run will do)
    done = sorted(tmp_path_factory.getbasetemp().glob("*/" + name + ".s"))
    out = done[0] if done else tmp_path_factory.mktemp("asm") / (name + ".s")
    if not done:
        proc = subprocess.run(["hipcc"] + FLAGS + SOURCES[name] + ["-o", str(out), os.path.join(CSRC, name)], stdout=subprocess.PIPE,
                              stderr=subprocess.STDOUT, text=True)
        assert proc.returncode == 0, proc.stdout[-2000:]
    text = out.read_text()
    assert asm_matrix_instructions(text)
    broken = broken_wait_states(text)
    assert not broken, f"{len(broken)} of them, first {broken[0]}"

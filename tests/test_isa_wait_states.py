"""Wait states around the kernels' inline assembly, which the compiler's hazard pass does not
look into: the batched kernels' gfx950 assembly (built here from their source) is read
instruction by instruction. The numbers are those the compiler itself inserts for gfx950.

  * after a store of more than 8 bytes, two wait states before a VALU write of its data
    registers (the store reads them late);
  * after an instruction that writes a part of a register (SDWA's dst_sel, op_sel's upper half),
    one before a VALU read of it, which keeping the register's other part is too.
"""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG, ROOT

REG = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")
PART_WRITE = re.compile(r"dst_sel:(WORD|BYTE)|op_sel:\[(\d,)+1\]")
WIDE_STORE = re.compile(r"(global|flat)_store_dwordx[34]")
TWO_DST = re.compile(r"v_(permlane\d+_swap|swap)_")


def _regs(text):
    out = set()
    for lo, hi, one in REG.findall(text):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def _operands(line):
    """Opcode and comma-separated operands (modifiers stay with the last one)."""
    op, _, rest = line.replace("\t", " ").partition(" ")
    return op, [o.strip() for o in re.split(r",(?![^\[]*\])", rest)]


def hazards(asm):
    """(line, writer, victim) of every pair of instructions with too few wait states between."""
    # pending: (registers, "write" or "read" that must wait, wait states still needed, line)
    bad, pending = [], []
    for n, line in enumerate(asm.splitlines(), 1):
        line = line.split(";")[0].strip()
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        op, args = _operands(line)
        if op in ("s_endpgm", "s_branch"):
            pending = []
            continue
        if op.startswith("v_"):
            first = 2 if TWO_DST.match(op) else 1
            dst, src = _regs(" ".join(args[:first])), _regs(" ".join(args[first:]))
            if "UNUSED_PRESERVE" in line or first == 2 or re.match(r"v_(fmac|mac|dot2c)_", op):
                src |= dst
            bad += [(n, was, line) for regs, how, _, was in pending
                    if regs & (dst if how == "write" else src)]
        states = int(args[0], 0) + 1 if op == "s_nop" else 1
        pending = [(r, how, left - states, was) for r, how, left, was in pending if left > states]
        if WIDE_STORE.match(op):
            pending.append((_regs(args[1]), "write", 2, line))
        if op.startswith("v_") and PART_WRITE.search(line):
            pending.append((dst, "read", 1, line))
    return bad


def test_reader_finds_a_short_wait():
    store = "global_store_dwordx4 v[2:3], v[4:7], off sc1\n s_nop %d\n v_mov_b32_e32 v5, v1\n"
    assert len(hazards(store % 0)) == 1 and not hazards(store % 1)
    assert not hazards((store % 0).replace("v5, v1", "v1, v5"))
    part = "v_add_f16_sdwa v4, v2, v2 dst_sel:WORD_%d dst_unused:UNUSED_%s src0_sel:WORD_1 src1_sel:WORD_0\n"
    pair = part % (0, "PAD"), part % (1, "PRESERVE")
    assert len(hazards("".join(pair))) == 1 and not hazards("v_mov_b32_e32 v1, v0\n".join(pair))
    assert len(hazards(pair[0] + "v_mov_b32_e32 v1, v4\n")) == 1


KERNELS = ["bgemm_kernel<3, CB_MCG, 1, 2, 0, false>", "bgemm_kernel<3, CB_MCG, 1, 4, 0, false>",
           "bgemm_wide_kernel<3, CB_MCG, 1, 8, 0, false>", "bgemm_wide_kernel<3, CB_MCG, 2, 8, 1, false>",
           "bgemm_wide_kernel<3, CB_3INST, 1, 16, 1, false>", "bgemm_kernel<4, CB_MCG, 1, 4, 1, true>",
           "bgemm_shared_kernel<3, CB_MCG, 1, 4, 1, false>"]


@pytest.mark.parametrize("kernel", KERNELS)
def test_kernel_wait_states(tmp_path, kernel):
    spec = importlib.util.spec_from_file_location("te_build", os.path.join(ROOT, PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if shutil.which(build.HIPCC) is None:
        pytest.skip("no hipcc")
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text('#include <hip/hip_runtime.h>\n#include "bgemm.h"\n'
                   "namespace trellis { template __global__ void %s(LinArgs); }\n" % kernel)
    subprocess.run([build.HIPCC, *build.FLAGS, "-w", "-I", os.path.join(ROOT, "include"), "-I", build.CSRC,
                    "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True)
    asm = out.read_text()
    assert "v_mfma" in asm
    bad = hazards(asm)
    assert not bad, f"{len(bad)} in {kernel}, first {bad[0]}"

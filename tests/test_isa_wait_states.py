"""Wait states around the kernels' inline assembly, which the compiler's hazard pass does not
look into: the batched kernels' gfx950 assembly (built here from their source) is read
instruction by instruction. The numbers are those the compiler itself inserts for gfx950.

  * after a store of more than 8 bytes, two wait states before a VALU write of its data
    registers (the store reads them late).
"""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG, ROOT

REG = re.compile(r"\bv(?:\[(\d+):(\d+)\]|(\d+)\b)")
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
    bad, pending = [], []          # pending: (registers, wait states still needed, line)
    for n, line in enumerate(asm.splitlines(), 1):
        line = line.split(";")[0].strip()
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        op, args = _operands(line)
        if op in ("s_endpgm", "s_branch"):
            pending = []
            continue
        if op.startswith("v_"):
            dst = _regs(" ".join(args[:2 if TWO_DST.match(op) else 1]))
            bad += [(n, was, line) for regs, _, was in pending if regs & dst]
        states = int(args[0], 0) + 1 if op == "s_nop" else 1
        pending = [(r, left - states, was) for r, left, was in pending if left > states]
        if WIDE_STORE.match(op):
            pending.append((_regs(args[1]), 2, line))
    return bad


def test_reader_finds_a_short_wait():
    store = "global_store_dwordx4 v[2:3], v[4:7], off sc1\n s_nop %d\n v_mov_b32_e32 v5, v1\n"
    assert len(hazards(store % 0)) == 1 and not hazards(store % 1)
    assert not hazards((store % 0).replace("v5, v1", "v1, v5"))


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

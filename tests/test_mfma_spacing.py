"""Distances around the hand-placed MFMAs of the prefill kernels (CPU, compiled code).

The tile-image kernels issue v_mfma through inline assembly, which the compiler
does not recognise as such, so it keeps none of the wait states an MFMA needs
against vector instructions.  This reads the AMD assembly of the kernels as
built here and checks them, counting every instruction as one state (and
``s_nop n`` as n + 1) within straight-line order:

* an operand written by a vector instruction is read two states later or more;
* a result is read or overwritten by anything but an MFMA accumulating into it
  18 states later or more (a 16-pass product's requirement).
"""
from __future__ import annotations

import re
import shutil
import subprocess

import pytest

from k8v4_v030 import _build

RESULT_STATES, OPERAND_STATES = 18, 2
KERNELS = ("prefill_tiles_kernelILi128", "prefill_tiles_kernelILi256")


def _regs(text):
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", text):
        if m.group(1):
            out |= {(m.group(1), k) for k in range(int(m.group(2)), int(m.group(3)) + 1)}
        else:
            out.add((m.group(4), int(m.group(5))))
    return out


def _violations(body):
    result, written, now, bad = {}, {}, 0, []
    for line in body.split("\n"):
        ins = line.split(";")[0].strip()
        if not ins or ins.startswith(".") or ins.endswith(":"):
            continue
        op = ins.split()[0]
        args = ins[len(op) :]
        if op == "s_nop":
            now += int(args) + 1
            continue
        now += 1
        if op.startswith("s_"):
            continue
        parts = re.split(r",(?![^\[]*\])", args)
        if op.startswith("v_mfma"):
            if any(now - result.get(r, -99) <= RESULT_STATES for p in parts[1:3] for r in _regs(p)):
                bad.append(ins)
            if any(now - written.get(r, -99) <= OPERAND_STATES for p in parts[1:4] for r in _regs(p)):
                bad.append(ins)
            for r in _regs(parts[0]):
                result[r] = now
                written.pop(r, None)
            continue
        if any(now - result.get(r, -99) <= RESULT_STATES for r in _regs(args)):
            bad.append(ins)
        if op.startswith("v_"):
            for r in _regs(parts[0]) | (_regs(parts[1]) if "swap" in op else set()):
                written[r] = now
    return bad


def test_the_check_sees_both_kinds():
    mfma = "v_mfma_f32_32x32x16_f16 v[0:15], a[0:3], a[4:7], v[0:15]\n"
    assert _violations("v_accvgpr_write_b32 a1, v40\ns_nop 0\n" + mfma)
    assert not _violations("v_accvgpr_write_b32 a1, v40\ns_nop 1\n" + mfma)
    assert _violations(mfma + "s_nop 15\nv_exp_f32_e32 v40, v3\n")
    assert not _violations(mfma + "s_nop 15\ns_nop 1\nv_exp_f32_e32 v40, v3\n")


@pytest.mark.skipif(shutil.which(_build.hipcc()) is None, reason="no hipcc")
def test_prefill_kernels_keep_the_distances(tmp_path):
    asm = tmp_path / "prefill.s"
    subprocess.run([_build.hipcc(), *_build.COMMON_FLAGS, *_build.PER_FILE_FLAGS["prefill.hip"], "-S",
                    "--cuda-device-only", str(_build.CSRC / "prefill.hip"), "-o", str(asm)],
                   check=True, capture_output=True)
    text = asm.read_text()
    for kernel in KERNELS:
        name = next(n for n in re.findall(r"^(\w+):", text, re.M) if kernel in n)
        start = text.index("\n%s:" % name)
        body = text[start : text.index(".Lfunc_end", start)]
        assert body.count("v_mfma_f32_32x32x16_f16") >= 160
        assert _violations(body) == []

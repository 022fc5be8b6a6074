"""Distances around the hand-placed MFMAs of the prefill kernels (CPU, compiled code).

The tile-image kernels issue v_mfma through inline assembly, which the compiler
does not recognise as such, so it keeps none of the wait states an MFMA needs
against vector instructions.  This reads the AMD assembly of the kernels as
built here and checks them on every path (branches and loops included), counting
every instruction as one state and ``s_nop n`` as n + 1:

* an operand written by a vector instruction is read two states later or more;
* a result is read or overwritten by anything but an MFMA accumulating into the
  same registers 18 states later or more (a 16-pass product's requirement);
* a start value in registers other than the result's is overwritten by a vector
  instruction 15 states later or more (likewise).
"""
from __future__ import annotations

import re
import shutil
import subprocess

import pytest

from k8v4_v030 import _build

RESULT_STATES, OPERAND_STATES, START_STATES = 18, 2, 15
KERNELS = ("prefill_tiles_kernelILi128", "prefill_tiles_kernelILi256")


def _regs(text):
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", text):
        if m.group(1):
            out |= {(m.group(1), k) for k in range(int(m.group(2)), int(m.group(3)) + 1)}
        else:
            out.add((m.group(4), int(m.group(5))))
    return out


def _blocks(body):
    """Basic blocks in file order: label, instructions, labels that may follow."""
    blocks = [["", [], []]]
    for line in body.split("\n"):
        ins = line.split(";")[0].strip()
        if re.fullmatch(r"\.LBB\w+:", ins):
            blocks.append([ins[:-1], [], []])
        elif ins and not ins.startswith(".") and not ins.endswith(":"):
            blocks[-1][1].append(ins)
            if ins.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                blocks[-1][2] += ins.split()[1:] if "branch" in ins else []
                blocks.append(["", [], []])
    for k, (_, code, after) in enumerate(blocks):
        if k + 1 < len(blocks) and not (code and code[-1].startswith(("s_branch", "s_endpgm"))):
            after.append(k + 1)
    at = {label: k for k, (label, _, _) in enumerate(blocks) if label}
    return [(code, [x if isinstance(x, int) else at[x] for x in after]) for _, code, after in blocks]


def _walk(code, state, bad):
    """One block from the states since (negative: before its start) each register's
    last product result {(register, tuple): state}, vector write and read as a
    product's start value; returns the same at its end."""
    result, written, started = (dict(x) for x in state)
    now = 0

    def within(seen, regs, states, but=""):
        return any(now - t <= states and k[1] != but for k, t in seen.items() if k[0] in regs)

    for ins in code:
        op = ins.split()[0]
        args = ins[len(op) :]
        if op == "s_nop":
            now += int(args) + 1
            continue
        now += 1
        if op.startswith("s_"):
            continue
        for seen, states in ((result, RESULT_STATES), (written, OPERAND_STATES), (started, START_STATES)):
            for k in [k for k, t in seen.items() if now - t > states]:
                del seen[k]
        parts = [p.strip() for p in re.split(r",(?![^\[]*\])", args)]
        if op.startswith("v_mfma"):
            dst, start = _regs(parts[0]), _regs(parts[3])
            if within(result, _regs(parts[1]) | _regs(parts[2]), RESULT_STATES):
                bad.append("result as operand: " + ins)
            if within(result, dst, RESULT_STATES, parts[0]) or within(result, start, RESULT_STATES, parts[3]):
                bad.append("result overlapped: " + ins)
            if within(written, dst | start | _regs(parts[1]) | _regs(parts[2]), OPERAND_STATES):
                bad.append("operand just written: " + ins)
            for r in dst:
                for k in [k for k in result if k[0] == r]:
                    del result[k]
                result[r, parts[0]] = now
            if parts[3] != parts[0]:
                started.update({(r, None): now for r in start})
            continue
        regs = _regs(args)
        if result and within(result, regs, RESULT_STATES):
            bad.append("result: " + ins)
        if op.startswith("v_"):
            dst = _regs(parts[0]) | (_regs(parts[1]) if "swap" in op else set())
            if started and within(started, dst, START_STATES):
                bad.append("start value overwritten: " + ins)
            written.update({(r, None): now for r in dst})
    return tuple({k: t - now for k, t in seen.items()} for seen in (result, written, started))


def _violations(body):
    """Over all paths: a block's entry state is the latest of those it may be reached with."""
    blocks = _blocks(body)
    entry = [({}, {}, {}) for _ in blocks]
    todo, bad = {0}, {}
    while todo:
        k = todo.pop()
        bad[k] = []
        end = _walk(blocks[k][0], entry[k], bad[k])
        for nxt in blocks[k][1]:
            grown = False
            for have, got in zip(entry[nxt], end):
                for key, t in got.items():
                    if have.get(key, -99) < t:
                        have[key] = t
                        grown = True
            if grown or nxt not in bad:
                todo.add(nxt)
    return [ins for k in sorted(bad) for ins in bad[k]]


def test_the_check_sees_every_kind():
    mfma = "v_mfma_f32_32x32x16_f16 v[0:15], a[0:3], a[4:7], v[0:15]\n"
    assert _violations("v_accvgpr_write_b32 a1, v40\ns_nop 0\n" + mfma)
    assert not _violations("v_accvgpr_write_b32 a1, v40\ns_nop 1\n" + mfma)
    assert _violations(mfma + "s_nop 15\nv_exp_f32_e32 v40, v3\n")
    assert not _violations(mfma + "s_nop 15\ns_nop 1\nv_exp_f32_e32 v40, v3\n")
    assert not _violations(mfma + mfma)
    # another product over a part of the result
    assert _violations(mfma + mfma.replace("v[0:15]", "v[8:23]"))
    # a start value overwritten while the product may still read it
    apart = mfma.replace(", v[0:15]", ", v[16:31]")
    assert _violations(apart + "s_nop 13\nv_mov_b32_e32 v17, v40\n")
    assert not _violations(apart + "s_nop 14\nv_mov_b32_e32 v17, v40\n")
    # across a loop's back edge and into a block placed elsewhere
    loop = ".LBB0_1:\nv_exp_f32_e32 v40, v3\ns_nop 15\n%s" + mfma + "s_cbranch_scc1 .LBB0_1\ns_endpgm\n"
    assert _violations(loop % "")
    assert not _violations(loop.replace("s_cbranch", "s_nop 15\ns_nop 1\ns_cbranch") % "")
    far = mfma + "s_cbranch_scc1 .LBB0_2\ns_nop 15\ns_nop 1\n.LBB0_1:\nv_exp_f32_e32 v40, v3\ns_endpgm\n.LBB0_2:\n%ss_branch .LBB0_1\n"
    assert _violations(far % "")
    assert not _violations(far % "s_nop 15\ns_nop 1\n")


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

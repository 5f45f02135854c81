"""The products of fp16 matrices read LDS with ds_read_b64_tr_b16 in inline assembly (gw_read_tr, gd_read_tr): the compiler
does not know that the result is there only behind the next wait for lgkmcnt.  A copy, a spill or a use that it put in
front of that wait would take what the register held before.  This walks the code that it makes of the two files, from every
such read along every branch to a wait for all LDS reads, and finds no instruction that names the read's registers."""
import os
import re
import shutil
import subprocess

import pytest

from helpers import ROOT

CSRC = os.path.join(ROOT, "occamy_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
READ = "ds_read_b64_tr_b16"


def _code(text):
    """The instructions of an assembly listing, and where its labels stand."""
    code, labels = [], {}
    for line in text.splitlines():
        line = re.sub(r"(;|//).*", "", line).strip()
        label = re.match(r"([.\w$]+):", line)
        if label:
            labels[label.group(1)] = len(code)
        elif line and not line.startswith("."):
            code.append(line)
    return code, labels


def _vgprs(text):
    regs = set()
    for lo, hi in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        regs.update(range(int(lo), int(hi) + 1))
    return regs | {int(n) for n in re.findall(r"\bv(\d+)\b", text)}


def _waits_for_lds(op):
    return op.startswith("s_waitcnt") and re.search(r"lgkmcnt\(0\)", op) is not None


def touched_early(text):
    """(number of reads, [(read, instruction in front of the wait that names its registers)])."""
    code, labels = _code(text)
    found, reads = [], 0
    for i, op in enumerate(code):
        if not op.startswith(READ):
            continue
        reads += 1
        mine = _vgprs(op.split(",")[0])
        todo, seen = [i + 1], set()
        while todo:
            at = todo.pop()
            if at in seen:
                continue
            seen.add(at)
            here = code[at]
            if _waits_for_lds(here):
                continue
            if here.startswith("s_endpgm") or _vgprs(here) & mine:  # an end without a wait: the value was not waited for at all
                found.append((op, here))
                continue
            branch = re.match(r"s_(c?)branch\w*\s+([.\w$]+)", here)
            if branch:
                todo.append(labels[branch.group(2)])
                if not branch.group(1):
                    continue
            todo.append(at + 1)
    return reads, found


@pytest.mark.parametrize("name", ["gemm_f16_waves", "gemm_f16_dma"])
def test_nothing_touches_a_transposing_read_in_front_of_its_wait(name, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    makefile = open(os.path.join(CSRC, "Makefile")).read().replace("\\\n", " ")
    flags = re.search(r"^HIPFLAGS\s*=\s*(.*)$", makefile, re.M).group(1).replace("$(ARCH)", "gfx950").split()
    out = tmp_path / "code.s"
    subprocess.check_call([HIPCC] + flags + ["--cuda-device-only", "-S", os.path.join(CSRC, name + ".hip"), "-o", str(out)], cwd=CSRC, stderr=subprocess.DEVNULL)
    reads, found = touched_early(out.read_text())
    assert reads >= 24 and not found


@pytest.mark.parametrize("tail,early", [
    ("s_waitcnt lgkmcnt(0)\n v_mov_b32_e32 v9, v4", False),
    ("s_waitcnt vmcnt(3) lgkmcnt(0)\n v_mov_b32_e32 v9, v4", False),
    ("v_mov_b32_e32 v9, v5\n s_waitcnt lgkmcnt(0)", True),
    ("s_waitcnt lgkmcnt(1)\n v_mov_b32_e32 v4, v9", True),
    ("scratch_store_dwordx2 off, v[4:5], off\n s_waitcnt lgkmcnt(0)", True),
    ("s_cbranch_scc1 .L2\n s_waitcnt lgkmcnt(0)\n s_endpgm\n.L2:\n v_mov_b32_e32 v9, v4", True),
    ("s_branch .L2\n v_mov_b32_e32 v9, v4\n.L2:\n s_waitcnt lgkmcnt(0)", False),
    ("s_endpgm", True),
])
def test_the_walk_sees_early_uses(tail, early):
    reads, found = touched_early("k:\n ds_read_b64_tr_b16 v[4:5], v2 offset:0 ; comment v4\n v_add_u32_e32 v3, v2, v1\n " + tail + "\n s_endpgm\n")
    assert reads == 1 and bool(found) == early

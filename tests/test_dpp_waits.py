"""Wait states of the FP64 M2L's row broadcasts (m2l_bcast_kernel.hpp) on every path.

A register that a vector instruction wrote may be read through DPP two wait
states later.  The products are inline assembly, which the compiler does not
check, so the built kernels are: every way that execution can reach a DPP read
is followed back through two wait states, over branches, skipped blocks and the
back edges of loops.
"""
import os
import re
import shutil
import subprocess

import pytest

from simplefmm_amd import api

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _registers(token):
    m = re.match(r"-?\|?v\[(\d+):(\d+)\]", token) or re.match(r"-?\|?v(\d+)", token)
    return set() if m is None else set(range(int(m[1]), int(m[m.lastindex]) + 1))


class _Instr:
    __slots__ = ("text", "states", "wrote", "reads", "falls", "came")

    def __init__(self, op, args, text):
        self.text = text
        self.states = int(args[0], 0) + 1 if op == "s_nop" else 1
        vector = op.startswith("v_") and not op.startswith("v_cmp")
        self.wrote = _registers(args[0]) if vector else set()
        self.reads = _registers(args[1]) if "row_newbcast" in text else None
        self.falls = op not in ("s_branch", "s_endpgm", "s_setpc_b64", "s_trap")
        self.came = []  # branches to this instruction


def hazards(listing):
    """(DPP reads, reads that some path reaches within two wait states of a vector
    write of the register) of an llvm-objdump listing with addresses."""
    code, at, jumps = [], {}, []
    for line in listing:
        m = re.match(r"\s+([a-z]+_\w+)\s*(.*?)\s*//\s*([0-9A-F]+):", line)
        if m is None:
            if re.match(r"[0-9a-f]+ <", line) and code:
                code[-1].falls = False  # another function
            continue
        args = [a.strip() for a in m[2].split(",")]
        pc = int(m[3], 16)
        if m[1] == "s_branch" or m[1].startswith("s_cbranch"):
            off = int(args[0], 0) & 0xFFFF
            jumps.append((len(code), pc + 4 + 4 * (off - 0x10000 if off >= 0x8000 else off)))
        at[pc] = len(code)
        code.append(_Instr(m[1], args, f"{m[1]} {m[2]}"))
    for source, target in jumps:
        code[at[target]].came.append(source)
    reads, bad = 0, []
    for i, ins in enumerate(code):
        if ins.reads is None:
            continue
        reads += 1
        todo = [(i, 0)]
        while todo:
            k, waits = todo.pop()
            before = list(code[k].came)
            if k > 0 and code[k - 1].falls:
                before.append(k - 1)
            for b in before:
                if code[b].wrote & ins.reads:
                    bad.append((code[b].text, ins.text))
                elif waits + code[b].states < 2:
                    todo.append((b, waits + code[b].states))
    return reads, bad


READ = "v_fmac_f64_dpp v[0:1], v[4:5], v[2:3] row_newbcast:3 row_mask:0xf"


def _listing(*lines):
    return [f"\t{text} // {0x100 + 4 * k:012X}: 00000000" for k, text in enumerate(lines)]


@pytest.mark.parametrize("lines,bad", [
    (["v_mov_b32_e32 v4, v9", "s_nop 0", READ], 1),
    (["v_mov_b32_e32 v4, v9", "s_nop 1", READ], 0),
    # the wait lies in a block that a branch skips
    (["v_mov_b32_e32 v4, v9", "s_cbranch_scc1 1", "s_nop 1", READ], 1),
    (["v_mov_b32_e32 v4, v9", "s_cbranch_scc1 1", "s_nop 1", "s_nop 0", READ], 0),
    # the write lies at the end of a loop, the read at its start
    (["s_nop 1", READ, "v_mov_b32_e32 v5, v9", "s_cbranch_scc1 65533"], 1),
    (["s_nop 1", READ, "v_mov_b32_e32 v5, v9", "s_cbranch_scc1 65532"], 0),
    (["s_nop 1", READ, "v_mov_b32_e32 v7, v9", "s_cbranch_scc1 65533"], 0),
    # no path from the write to the read
    (["v_mov_b32_e32 v4, v9", "s_endpgm", READ], 0),
], ids=["near", "far", "skipped", "after_skip", "back_edge", "back_edge_waits", "other_register", "no_path"])
def test_planted_hazards_are_seen(lines, bad):
    reads, found = hazards(_listing(*lines))
    assert reads == 1 and len(found) == bad


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(api.LIB_PATH)), reason="needs the built library")
def test_built_kernels_wait_on_every_path(tmp_path):
    lib = shutil.copy(api.LIB_PATH, tmp_path / "libsfmm.so")
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    reads = 0
    for name in sorted(os.listdir(tmp_path)):
        if "gfx950" not in name:
            continue
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / name)], check=True,
                             capture_output=True, text=True).stdout
        if "row_newbcast" not in out:
            continue
        n, bad = hazards(out.splitlines())
        reads += n
        assert not bad, (name, len(bad), bad[:3])
    assert reads > 10000

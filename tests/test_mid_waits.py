"""The hand-counted waits of moe_mid_kernel, read from the assembly that its source compiles to.

A stage of its k-loop waits until at most 8 vector memory operations are in flight and takes the activation copies into LDS of
the stage before as landed. That holds only if every such copy is issued before at least 8 later vector memory operations;
nothing at run time would show a compiler that reordered them (LDS read too early gives wrong sums now and then), so the order
is checked here. CPU only: hipcc cross-compiles the one file.
"""

from __future__ import annotations

import re
import shutil
import subprocess

import pytest

from cernels_amd import build

STAGE_WAIT = 8


def _kernels(text):
    return {m.group(1): m.group(2).splitlines()
            for m in re.finditer(r"^(_ZN4cmoe14moe_mid_kernel\S+):.*?\n(.*?)\.Lfunc_end", text, re.S | re.M)}


def _issue_order(lines):
    """'copy' (into LDS), 'load' (to registers), 'wait' and 'barrier' in program order."""
    out = []
    for ln in lines:
        op = ln.strip()
        if re.match(r"(buffer|global)_load", op):
            out.append("copy" if re.search(r"\blds\b", op) or "load_lds" in op else "load")
        elif op.startswith("s_waitcnt") and f"vmcnt({STAGE_WAIT}) lgkmcnt(0)" in op:
            out.append("wait")
        elif op.startswith("s_barrier"):
            out.append("barrier")
    return out


def _copies_without_loads(ops):
    """Stage waits (directly before a barrier) that fewer than STAGE_WAIT loads separate from the copies they stand for."""
    bad, since = [], None
    for i, op in enumerate(ops):
        if op == "copy":
            since = 0
        elif op == "load" and since is not None:
            since += 1
        elif op == "wait" and i + 1 < len(ops) and ops[i + 1] == "barrier" and (since is None or since < STAGE_WAIT):
            bad.append((i, since))
    return bad


def test_checker_sees_a_hoisted_load():
    good = ["copy"] * 4 + ["load"] * 8 + ["wait", "barrier"] + ["copy"] * 4 + ["load"] * 8 + ["wait", "barrier"]
    assert not _copies_without_loads(good)
    hoisted = ["load"] + ["copy"] * 4 + ["load"] * 7 + ["wait", "barrier"]
    assert _copies_without_loads(hoisted)


@pytest.mark.skipif(shutil.which(build.HIPCC) is None, reason="hipcc not available")
def test_stage_copies_are_issued_before_the_loads_that_cover_them(tmp_path):
    asm = tmp_path / "stream.s"
    cmd = [build.HIPCC, *build.COMMON, "-x", "hip", *build.DEVICE, "--cuda-device-only", "-S",
           str(build.CSRC / "moe_stream.hip"), "-o", str(asm)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    kernels = _kernels(asm.read_text())
    assert len(kernels) == 8, sorted(kernels)  # two gated activations with and without bias, three plain ones, down
    for name, lines in kernels.items():
        ops = _issue_order(lines)
        assert ops.count("wait") >= 8, name  # two stages in each of the four row-block forms
        assert not _copies_without_loads(ops), name

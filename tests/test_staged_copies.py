"""Copies from memory straight to LDS (global_load_lds) land some time after they
are issued, and no language rule ties them to a barrier: the wave that issued them
must have waited for them (vmcnt(0)) before the barrier that hands them to others.
Checked in the source (the wait stands before the barrier) and in the code that the
library's own flags give for every instance. Needs hipcc, no GPU."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from crosslane_amd import _build

SRC = os.path.join(_build.CSRC, "xl_shared.hip")


def test_the_source_waits_before_the_step_barrier():
    text = re.sub(r"//[^\n]*", "", open(SRC).read())
    loop = text[text.index("for (int s = 0; s < steps; ++s)"):]
    before = loop[:loop.index("__syncthreads();")]
    assert "__builtin_amdgcn_s_waitcnt(vmcnt_imm(0));" in before and "stage_step" not in before


def test_no_barrier_with_copies_in_flight(tmp_path):
    if not shutil.which(_build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path / "shared.s")
    subprocess.run([_build.HIPCC, *_build.CFLAGS, "-w", "--cuda-device-only", "-S", SRC, "-o", out], check=True)
    kernels, name, pending, staged = 0, None, False, 0
    for line in open(out):
        m = re.match(r"(_Z\w*ffn_\w*):", line)
        if m:
            kernels, name, pending = kernels + 1, m.group(1), False
        elif line.startswith("\t.section") or line.startswith(".Lfunc_end"):
            name = None
        elif name and re.search(r"\b(global|buffer)_load_lds", line):
            pending, staged = True, staged + 1
        elif name and "s_waitcnt" in line and "vmcnt(0)" in line:
            pending = False
        elif name and "s_barrier" in line:
            assert not pending, (name, line)
    assert kernels == 16 and staged >= 2 * kernels      # two forms of gate/up and of down by four formats

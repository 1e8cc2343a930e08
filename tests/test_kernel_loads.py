"""Loads of the step kernels in the built library's gfx950 code: the
instantiations that read the operator through the caches hold no streaming
load, those that stream it do."""
import os
import re
import shutil
import subprocess

import pytest

from lymph3d_apsc_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# k_leapfrog<P, MODE, ..., NT>, k_leapfrog32, k_leapfrog48, k_leapfrog_packed, k_leapfrog_joint
STEP = re.compile(r"^<_ZN5lymph\d+(k_leapfrog(?:32|48|_packed|_joint)?)I((?:Li\d+E)+)Lb([01])EEEv.*>:$")


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(_lib.LIB_PATH)), reason="no disassembler or library")
def test_cached_step_kernels_hold_no_streaming_loads(tmp_path):
    so = shutil.copy(_lib.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", so], cwd=tmp_path, check=True, capture_output=True)
    code = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert len(code) == 1, code
    asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", tmp_path / code[0]], check=True,
                         capture_output=True, text=True).stdout
    seen, kernel = {}, None
    for line in asm.splitlines():
        if line.endswith(">:"):
            m = STEP.match(line)
            kernel = None
            if m:
                kernel = (m[1], tuple(map(int, re.findall(r"\d+", m[2]))), m[3] == "1")
                seen[kernel] = [0, 0]
        elif kernel and "global_load" in line:
            seen[kernel][bool(re.search(r" nt\b", line))] += 1
    assert {k[0] for k in seen} == {"k_leapfrog" + s for s in ("", "32", "48", "_packed", "_joint")}
    for (name, args, nt), (cached, streaming) in seen.items():
        assert cached > 0 and (streaming > 0) == nt, (name, args, nt, cached, streaming)

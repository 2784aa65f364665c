"""CPU: the topology's pass A kernel (zedm-x_amd/csrc/zdx_pass_a.h) compiled for
the host under the SIMT emulation with AddressSanitizer and
UndefinedBehaviorSanitizer, against the serial tests it stands for
(tests/csrc/pass_a_emu.cpp): rows, longest row and snap words, all equal."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pass_a_under_simt_emulation(tmp_path):
    exe = str(tmp_path / "pass_a_emu")
    cmd = ["g++", "-std=c++17", "-O0", "-g", "-fno-omit-frame-pointer", "-ffp-contract=off",
           "-fsanitize=address,undefined", "-fno-sanitize=float-cast-overflow", "-fwrapv", "-fno-sanitize-recover=all", "-w",
           "-o", exe, os.path.join(ROOT, "tests", "csrc", "pass_a_emu.cpp")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, (r.stdout[-3000:], r.stderr[-4000:])
    assert "pass_a_emu ok" in r.stdout

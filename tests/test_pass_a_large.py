"""CPU: pass A's pair numbers where 32 bits end (tests/csrc/pass_a_large_emu.cpp):
pairs of 23300 and 32900 segments, whose endpoint pairs number up to 2.2e9, under
the SIMT emulation with signed overflow trapped.  And the larger workgroups of a
step's larger pairs, which give the rows and words of the smaller."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pass_a_pair_numbers_past_32_bits(tmp_path):
    exe = str(tmp_path / "pass_a_large_emu")
    r = subprocess.run(["g++", "-std=c++17", "-O0", "-g", "-ffp-contract=off", "-fsanitize=undefined",
                        "-fno-sanitize-recover=all", "-w", "-o", exe,
                        os.path.join(ROOT, "tests", "csrc", "pass_a_large_emu.cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, (r.stdout[-3000:], r.stderr[-4000:])
    assert "pass_a_large ok" in r.stdout

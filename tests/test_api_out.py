"""CPU: where the per-pair call's output arrays go (tests/csrc/api_out.cpp):
never through a null pointer, never past a buffer, nowhere when the caller's
array is too small."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_outputs_have_a_place_on_both_sides_of_the_slot(tmp_path):
    exe = str(tmp_path / "api_out")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                        "-Wall", "-o", exe, os.path.join(ROOT, "tests", "csrc", "api_out.cpp")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "api_out ok: 405" in r.stdout, (r.stdout, r.stderr)

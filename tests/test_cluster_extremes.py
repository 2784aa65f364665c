"""CPU: the cluster kernels at the ends of their range, under the SIMT emulation
(tests/csrc/cluster_extremes_emu.cpp): quaternions of norm 1e-14 and beside it
(the transform takes shorter ones for the identity) and past 1e154 (its norm
overflows, so it takes them for zero), and world vertices that are no numbers or
infinite."""
import os
import re
import shutil
import struct
import subprocess

import numpy as np
import pytest

from zdx import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def write_input(path, scales, n):
    meshes = [synth.icosphere(2), synth.star_mesh(3, 2)]
    rng = np.random.default_rng(7)
    out = [struct.pack("<i", len(meshes))]
    for m in meshes:
        out.append(struct.pack("<i", len(m)) + np.ascontiguousarray(m, "<f8").tobytes())
    out.append(struct.pack("<i", n))
    for k in range(n):
        d = rng.normal(size=3)
        d *= 0.9 / np.linalg.norm(d)
        for side in range(2):
            q = rng.normal(size=4)
            q *= scales[(2 * k + side) % len(scales)] / np.linalg.norm(q)
            out.append(struct.pack("<i", (k + side) % 2) + np.concatenate([d * side, q]).astype("<f8").tobytes())
    with open(path, "wb") as fh:
        fh.write(b"".join(out))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_extremes_under_simt_emulation(tmp_path):
    exe = str(tmp_path / "extremes")
    r = subprocess.run(["g++", "-std=c++17", "-O0", "-g", "-fno-omit-frame-pointer", "-ffp-contract=off",
                        "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-w", "-o", exe,
                        os.path.join(ROOT, "tests", "csrc", "cluster_extremes_emu.cpp"),
                        os.path.join(ROOT, "zedm-x_amd", "csrc", "zdx_host.cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    e = np.float64(1e-14)
    around = [e, np.nextafter(e, 0), np.nextafter(e, 1), 0.9e-14, 3e-15, 1e-100, 1.0]
    for scales, n, first in ((around, 12, 12), ([1e160, 1.0, 1e200, 7.0], 8, 8), ([1.0], 9, 0)):
        inp = str(tmp_path / "in.bin")
        write_input(inp, scales, n)
        r = subprocess.run([exe, inp, str(first)], capture_output=True, text=True, timeout=600)
        print(r.stdout)
        assert r.returncode == 0 and "cluster_extremes ok" in r.stdout, (r.stdout[-3000:], r.stderr[-3000:])
        assert int(re.search(r"(\d+) hits", r.stdout).group(1)) > 100

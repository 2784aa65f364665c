"""CPU: the narrow phase's cluster kernels (zedm-x_amd/csrc/zdx_cluster.h)
compiled for the host under the SIMT emulation with AddressSanitizer and
UndefinedBehaviorSanitizer, against a plain restatement (see
tests/csrc/cluster_emu.cpp): box tests, hits and segments of every pair, the
segments bit for bit in (ta, tb) order.  The pairs cover meshes at the edges
of a cluster (4, 12, 16 and 17 triangles), pairs without kept triangles,
kept triangles past a wave's and the largest workgroup's LDS, more hits than a
wave's list, and bodies far from the origin."""
import os
import re
import shutil
import struct
import subprocess

import numpy as np
import pytest

from zdx import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def fan(n):
    """A closed double cone over an n-gon: 2 n triangles."""
    a = 2 * np.pi * np.arange(n) / n
    r = np.stack([np.cos(a), np.sin(a), 0 * a], 1)
    t = [(r[k], r[(k + 1) % n], np.array([0, 0, s])) for k in range(n) for s in (0.8, -0.8)]
    return np.array([x if x[2][2] > 0 else (x[1], x[0], x[2]) for x in t], float)


def write_input(path):
    wavy = synth.icosphere(4).reshape(-1, 3)
    wavy = (wavy * (1 + 0.12 * np.cos(9 * wavy[:, :1]) * np.cos(9 * wavy[:, 1:2]))).reshape(-1, 3, 3)
    tetra = synth.convex_hull_mesh(np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1.0]]))
    meshes = {"tetra": tetra, "box": synth.box_wall(1.6, 1.6, 1.6), "fan16": fan(8), "fan18": fan(9),
              "ico1": synth.icosphere(1), "ico2": synth.icosphere(2), "ico3": synth.icosphere(3),
              "star": synth.star_hull_mesh(3, 642), "wavy": wavy}
    names = list(meshes)
    rad = {k: np.max(np.linalg.norm(v.reshape(-1, 3), axis=1)) for k, v in meshes.items()}
    cases = [("tetra", "tetra", 0.5), ("tetra", "box", 0.6), ("box", "box", 0.7), ("fan16", "fan18", 0.8),
             ("fan18", "fan18", 0.5), ("fan16", "ico1", 0.9), ("ico1", "ico2", 0.9), ("ico1", "ico2", 0.5),
             ("ico2", "ico2", 0.95), ("ico2", "ico2", 0.2), ("ico2", "ico1", 1.6), ("ico3", "ico3", 0.97),
             ("ico3", "ico3", 0.7), ("ico2", "ico2", 0.0), ("star", "ico3", 0.8), ("box", "ico3", 0.3),
             ("ico3", "tetra", 0.9), ("wavy", "wavy", 0.9), ("wavy", "box", 0.4),
             ("star", "wavy", 0.3)]
    rng = np.random.default_rng(11)
    out = [struct.pack("<i", len(names))]
    for k in names:
        out.append(struct.pack("<i", len(meshes[k])) + np.ascontiguousarray(meshes[k], "<f8").tobytes())
    out.append(struct.pack("<i", len(cases)))
    for n, (a, b, f) in enumerate(cases):
        d = rng.normal(size=3)
        d /= np.linalg.norm(d)
        base = rng.uniform(-5, 5, 3) * (1000.0 if n % 7 == 3 else 1.0)
        for m, c in ((a, base), (b, base + d * (rad[a] + rad[b]) * f)):
            q = rng.normal(size=4)   # normalised by the transform
            out.append(struct.pack("<i", names.index(m)) + np.concatenate([c, q]).astype("<f8").tobytes())
    with open(path, "wb") as fh:
        fh.write(b"".join(out))
    return len(cases)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_cluster_kernels_under_simt_emulation(tmp_path):
    exe = str(tmp_path / "cluster_emu")
    cmd = ["g++", "-std=c++17", "-O0", "-g", "-fno-omit-frame-pointer", "-ffp-contract=off",
           "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-w", "-o", exe,
           os.path.join(ROOT, "tests", "csrc", "cluster_emu.cpp"),
           os.path.join(ROOT, "zedm-x_amd", "csrc", "zdx_host.cpp")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    inp = str(tmp_path / "pairs.bin")
    n = write_input(inp)
    r = subprocess.run([exe, inp], capture_output=True, text=True, timeout=900,
                       env=dict(os.environ, UBSAN_OPTIONS="print_stacktrace=1"))
    print(r.stdout)
    assert r.returncode == 0, (r.stdout[-3000:], r.stderr[-4000:])
    assert "cluster_emu ok" in r.stdout
    m = re.search(r"most segments (\d+), most hits (\d+), most kept triangles (\d+), pairs without tests (\d+)", r.stdout)
    # several rounds of 64 segments; past the lists of a wave (512 hits, 231
    # kept triangles) and of the largest workgroup (1739); pairs without a test
    assert int(m.group(1)) > 256 and int(m.group(2)) > 512 and int(m.group(3)) > 1739 and int(m.group(4)) > 0
    left = [int(x) for x in re.findall(r"^ok wave\+group .*\((\d+) to the workgroup kernel\)", r.stdout, re.M)]
    assert len(left) == 4 and all(0 < x < n for x in left)

"""GPU: the broad phase of at most 256 particles (one workgroup, every pair
tested) against the reference's pair test (src/main.cpp:2049-2059), and against
the cell-binned broad phase: the same bodies among enough far ones to take
that path must have the same pairs and, after some steps, the same state, bit
for bit."""
import numpy as np
import pytest

from test_gpu_broadphase import all_pairs, exact_pairs
from zdx import synth
from zdx import workloads as W

zdx = pytest.importorskip("zdx")
pytestmark = pytest.mark.gpu


def workload(n, far, seed):
    """n hulls in a crowded cube, then `far` ones on a line that touch nothing."""
    g = np.random.Generator(np.random.PCG64(seed))
    small = synth.sphere_hull(32, seed)
    r = W._centred_radius(small)
    pos = g.uniform(0, 1e-3 * max(1.0, 0.8 * n ** (1 / 3)), size=(n, 3))
    line = np.stack([0.05 + 0.004 * np.arange(far), np.zeros(far), np.zeros(far)], 1)
    q = g.normal(size=(n + far, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    init = np.concatenate([np.concatenate([pos, line]), q, np.zeros((n + far, 6))], axis=1)
    mat = np.tile(np.array([2500.0, 1e6, 0.25, 0.5, 0.5]), (n + far, 1))
    return W.Workload("crowd", [small], ["hull32"], np.zeros(n + far, int), np.full(n + far, round(0.5e-3 / r, 6)), init,
                      mat, [], (0.0, 0.0, -9.81), 1e-6, 20, True)


@pytest.mark.parametrize("n", [1, 2, 5, 63, 64, 65, 255, 256])
def test_small_broad_phase(n):
    ctx = zdx.Context(0)
    sims = [W.build_sim(ctx, workload(n, far, 3 + n))[0] for far in (0, 257 - n + 3)]
    s = sims[0].state()
    rad = np.array([ctx.mesh_props[m][4] for m in sims[0].mesh_id])
    want = exact_pairs(s[:, :3], rad, all_pairs(n))
    assert n < 63 or len(want) > n
    for mode in (zdx.MODE_BATCHED, zdx.MODE_PLAIN):
        for k in range(4):
            c = [sim.step(1, mode) for sim in sims]
            assert c[0]["contacts"] == c[1]["contacts"] and c[0]["pairs"] == c[1]["pairs"]
            got = [sim.pairs() for sim in sims]
            if k == 0 and mode == zdx.MODE_BATCHED:
                assert np.array_equal(got[0], want), (len(got[0]), len(want))
            assert np.array_equal(got[0], got[1])
            a, b = sims[0].state(), sims[1].state()[:n]
            assert np.array_equal(a.view(np.int64), b.view(np.int64))
    ctx.close()

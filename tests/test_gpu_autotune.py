"""GPU: the autotuner on the cluster path.  A simulation that gives every pair a
workgroup at once (64 bodies and fewer) keeps its shape, and so does one whose
shape no other beats; shapes differ in threads and workgroups only, since these
kernels have no tests per thread; and no result depends on any of it."""
import numpy as np
import pytest

import zdx
from zdx import workloads as W

pytestmark = pytest.mark.gpu


def test_few_pairs_keep_their_shape():
    ctx = zdx.Context(0)
    sim, _ = W.build_sim(ctx, W.drop_on_plane(40, 3, height=-0.3e-3, gap=-0.35e-3))
    sim.step(3, zdx.MODE_BATCHED)
    for shape in ((12808, 4), (51202, 16)):
        sim.set_tiles(*shape)
        assert sim.autotune() == shape
    ctx.close()


def test_autotuned_shapes_and_results():
    out = []
    for tuned in (False, True):
        ctx = zdx.Context(0)
        sim, _ = W.build_sim(ctx, W.granular_bed(2000, seed=4, box=0.06, speed=0.8))
        sim.step(60, zdx.MODE_PLAIN)
        if tuned:
            block, groups = sim.autotune()
            assert block in (6404, 12804, 25604, 51204) and groups in (4, 8, 16)
            sim.set_tiles(block, groups)
        sim.step(40, zdx.MODE_BATCHED)
        out.append(sim.state().tobytes())
        ctx.close()
    assert out[0] == out[1]

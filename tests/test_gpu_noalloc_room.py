"""GPU: how much the 256 MiB of the no-allocation call hold: batches of 58500
pairs apart, 5200 overlapping boxes and 440 overlapping spheres of 1280
triangles fit, with the bytes of the allocating call."""
import numpy as np
import pytest

import zdx
from zdx import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh,n,dist", [("box", 58500, 3.0), ("box", 5200, 0.9), ("ball", 440, 1.2)])
def test_batches_that_fit(mesh, n, dist):
    ctx = zdx.Context(0)
    m = ctx.register_mesh(synth.box_wall(1.0, 1.0, 1.0) if mesh == "box" else synth.icosphere(3))
    ids, e, d = np.full(n, m), np.tile([1.0, 0.0, 0.0, 0.0], (n, 1)), np.zeros((n, 3))
    d[:, 0] = dist
    want = ctx.contact_pairs(ids, ids, np.zeros((n, 3)), e, d, e, vertices=False)
    got = ctx.contact_pairs(ids, ids, np.zeros((n, 3)), e, d, e, vertices=False, noalloc=True)
    for k in want:
        assert got[k].tobytes() == want[k].tobytes(), k
    ctx.close()

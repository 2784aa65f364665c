"""GPU: meshes registered between calls.  A shape's clusters are made once, at
the call after its first mesh, so a call after one more small mesh costs a
fraction of the first; and the results are those of a context that had all the
meshes at once."""
import time

import numpy as np
import pytest

import zdx
from zdx import synth

pytestmark = pytest.mark.gpu


def call(ctx, a, b):
    n = len(a)
    e = np.tile([1.0, 0.0, 0.0, 0.0], (n, 1))
    d = np.zeros((n, 3))
    d[:, 0] = np.linspace(0.8, 1.7, n)
    return ctx.contact_pairs(a, b, np.zeros((n, 3)), e, d, e, segments=True)


def test_shapes_are_clustered_once():
    rng = np.random.default_rng(2)
    ball = synth.icosphere(4)
    big = [ball[rng.permutation(len(ball))] for _ in range(60)]   # 60 orders of its triangles: 60 shapes
    small = [synth.sphere_hull(24 + k, k) for k in range(5)]
    ctx = zdx.Context(0)
    first = ctx.register_mesh(small[0])
    call(ctx, [first], [first])       # kernels loaded, buffers made
    ids = [ctx.register_mesh(m) for m in big]
    t = time.perf_counter()
    call(ctx, ids[:4], ids[4:8])
    once = time.perf_counter() - t
    again = []
    for m in small[1:]:
        ids.append(ctx.register_mesh(m))
        t = time.perf_counter()
        call(ctx, [first], [ids[-1]])
        again.append(time.perf_counter() - t)
    print(f"[register] call after 60 meshes {1e3 * once:.2f} ms, after one more {1e3 * min(again):.2f} ms", flush=True)
    # making the clusters took nine tenths of the first of these calls
    assert min(again) < 0.5 * once
    a, b = ids[:8] + ids[-2:], ids[8:16] + [ids[3], first]
    got = call(ctx, a, b)
    other = zdx.Context(0)
    every = [other.register_mesh(m) for m in [small[0]] + big + small[1:]]
    assert every == [first] + ids
    want = call(other, a, b)
    for k in want:
        assert got[k].tobytes() == want[k].tobytes(), k
    ctx.close()
    other.close()

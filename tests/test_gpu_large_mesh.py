"""GPU: a registered mesh of more than 65535 triangles sends every pair of its
context through the hit-arena kernels (zdx_narrow.h).  They give the bytes of the
cluster kernels: in calls of one to a thousand pairs, both modes, with
sensitivities, without allocation and from tiny buffers, in a simulation whose
context gets such a mesh between two steps; and the pair of the large mesh
itself is the oracle's."""
import os

import numpy as np
import pytest

import oracle as O
import zdx
from zdx import synth
from zdx import workloads as W

pytestmark = pytest.mark.gpu

LARGE = synth.icosphere(6)   # 81920 triangles


def batch(ids, pairs):
    return [np.array([ids[p[0]] for p in pairs]), np.array([ids[p[1]] for p in pairs])] + \
        [np.array([p[k] for p in pairs]) for k in (2, 3, 4, 5)]


@pytest.mark.parametrize("n,kw,tiny", [
    (1, dict(segments=True), False), (300, dict(segments=True, mode=zdx.MODE_PLAIN), False),
    (1000, dict(segments=True), False), (80, dict(segments=True, sensitivities=True), False),
    (120, dict(segments=True, noalloc=True), False), (64, dict(segments=True), True),
])
def test_calls_beside_a_large_mesh(n, kw, tiny):
    meshes, _, pairs = W.uneven_pairs(n, seed=n)
    want = None
    for large in (False, True):
        if tiny and large:
            os.environ["ZDX_START_CAPACITY"] = "tiny"
        try:
            ctx = zdx.Context(0)
        finally:
            os.environ.pop("ZDX_START_CAPACITY", None)
        ids = [ctx.register_mesh(m) for m in meshes]
        if large:
            ctx.register_mesh(LARGE)
        if kw.get("noalloc"):
            ctx.contact_pairs(*batch(ids, pairs[:1]))   # uploads the meshes
        got = ctx.contact_pairs(*batch(ids, pairs), **kw)
        again = ctx.contact_pairs(*batch(ids, pairs), **kw)   # in the buffers of the first
        want = want or got
        for k in want:
            assert got[k].tobytes() == want[k].tobytes() and again[k].tobytes() == want[k].tobytes(), (large, k)
        ctx.close()


def test_pair_of_the_large_mesh():
    ctx = zdx.Context(0)
    box = synth.box_wall(0.9, 0.8, 0.7)
    a, b = ctx.register_mesh(LARGE), ctx.register_mesh(box)
    q = np.array([0.9, 0.2, -0.3, 0.1])
    q /= np.linalg.norm(q)
    e, d = np.array([1.0, 0.0, 0.0, 0.0]), np.array([0.9, 0.35, 0.2])
    r = ctx.contact_pairs([a], [b], [np.zeros(3)], [e], [d], [q], segments=True)
    ta, pa, _ = O.build_mesh(LARGE)
    tb, _, _ = O.build_mesh(box)
    ref = O.pair_contact(ta, tb, np.zeros(3), e, d, q, pa[5], pa[6])
    assert len(ref["segments"]) > 100 and r["segments"].tobytes() == np.ascontiguousarray(ref["segments"]).tobytes()
    assert len(r["loops"]) == len(ref["loops"])
    assert np.array_equal(r["loops"][:, :13], ref["loops"][:, :13])
    ctx.close()


@pytest.mark.parametrize("scene,mode", [("drop", zdx.MODE_BATCHED), ("bed", zdx.MODE_BATCHED), ("bed", zdx.MODE_PLAIN)])
def test_simulation_whose_context_gets_a_large_mesh(scene, mode):
    out = []
    for large in (False, True):
        ctx = zdx.Context(0)
        wl = W.drop_on_plane(40, 3, height=-0.3e-3, gap=-0.35e-3) if scene == "drop" else \
            W.granular_bed(1500, seed=4, box=0.055, speed=0.8)
        sim, _ = W.build_sim(ctx, wl)
        total = {}
        for k in range(6):
            if large and k == 2:
                ctx.register_mesh(LARGE)
            if large and k == 4:
                ctx.register_mesh(synth.icosphere(1))
            c = sim.step(10, mode)
            total = {f: total.get(f, 0) + c[f] for f in ("contacts", "segments", "loops", "tri_checks")}
        F, T, n = sim.forces()
        out.append((sim.state().tobytes(), F.tobytes(), T.tobytes(), n.tobytes(), total))
        ctx.close()
    assert out[0] == out[1] and out[0][4]["contacts"] > 0

"""GPU: the per-pair call whose output exceeds both the caller's array and the
512 KiB slot of the call's pinned memory reports ZDX_CAPACITY with the totals,
and the retry gives the bytes that arrays large enough at once give: segments
past 10922, loop vertices past 21845, each with a first capacity below that."""
import ctypes as C

import numpy as np
import pytest

import zdx
from zdx import synth

pytestmark = pytest.mark.gpu


def pairs(ctx, n):
    """Overlapping fine spheres: each pair's intersection is one ring of more
    than 100 segments."""
    m = ctx.register_mesh(synth.icosphere(4))
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    q = rng.normal(size=(2, n, 4))
    q /= np.linalg.norm(q, axis=2, keepdims=True)
    ids = np.full(n, m)
    return ids, ids, np.zeros((n, 3)), q[0], d * rng.uniform(0.9, 1.2, (n, 1)), q[1]


def raw(ctx, p, loops, vtx, segs, noalloc=False):
    """The call into arrays of the given rows (0 segments: not asked for)."""
    n = len(p[0])
    rec = np.zeros(n, dtype=zdx.PAIR_IN_DTYPE)
    rec["mesh_a"], rec["mesh_b"], rec["pos_a"], rec["quat_a"], rec["pos_b"], rec["quat_b"] = p
    opts = zdx.ContactOpts(1, zdx.MODE_BATCHED, 1.0, 0, 0, 0.0)
    a = dict(lo=np.zeros(n + 1, np.int32), so=np.zeros(n + 1, np.int32), rec=np.zeros((loops, 28)),
             vo=np.zeros(loops + 1, np.int32), vtx=np.zeros((vtx, 3)), seg=np.zeros((max(segs, 1), 6)))
    out = zdx.PairOut(loop_offset=a["lo"].ctypes.data, seg_offset=a["so"].ctypes.data, loop_rec=a["rec"].ctypes.data,
                      loop_cap=loops, vtx_offset=a["vo"].ctypes.data, loop_vtx=a["vtx"].ctypes.data, vtx_cap=vtx,
                      segments=a["seg"].ctypes.data if segs else None, seg_cap=segs)
    fn = zdx.lib().zdx_contact_pairs_noalloc if noalloc else zdx.lib().zdx_contact_pairs
    return fn(ctx.h, rec.ctypes.data, n, C.byref(opts), C.byref(out)), out, a


@pytest.mark.parametrize("n,segments,noalloc", [(150, True, False), (150, True, True), (300, False, False)])
def test_retry_past_the_slot_gives_the_same_bytes(n, segments, noalloc):
    ctx = zdx.Context(0)
    p = pairs(ctx, n)
    room = 512 * n
    st, out, want = raw(ctx, p, 64 * n, room, room if segments else 0)
    assert st == zdx.OK
    nl, nv, ns = out.n_loops_total, out.n_vtx_total, out.n_seg_total
    print(f"[api out] {n} pairs: {nl} loops, {nv} vertices, {ns} segments", flush=True)
    # the totals are past the slots, the first guess of Context.contact_pairs is not
    assert ns > 10922 >= 64 * n or nv > 21845 >= 64 * n
    st, out, got = raw(ctx, p, 4 * n, 64 * n, 64 * n if segments else 0, noalloc)
    assert st == zdx.CAPACITY
    assert (out.n_loops_total, out.n_vtx_total) == (nl, nv) and (not segments or out.n_seg_total == ns)
    assert not (got["rec"].any() or got["vtx"].any() or got["seg"].any())
    r = ctx.contact_pairs(*p, segments=segments, noalloc=noalloc)
    assert r["loops"].tobytes() == want["rec"][:nl].tobytes()
    assert r["loop_vtx"].tobytes() == want["vtx"][:nv].tobytes()
    assert r["loop_offset"].tobytes() == want["lo"].tobytes()
    assert r["vtx_offset"].tobytes() == want["vo"][:nl + 1].tobytes()
    if segments:
        assert r["segments"].tobytes() == want["seg"][:ns].tobytes()
        assert r["seg_offset"].tobytes() == want["so"].tobytes()
    ctx.close()

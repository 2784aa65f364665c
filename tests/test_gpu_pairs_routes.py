"""GPU: the per-pair call gives a pair the same bytes whatever the size of the
call it is in: sizes around the calls packed by one workgroup (64 pairs), the
calls with a workgroup per pair (512), the pinned input (6900 pairs) and the
output slots (512 KiB per array, 65535 pairs of columns), in both modes, with
and without sensitivities and device allocation."""
import numpy as np
import pytest

import zdx
from zdx import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base():
    ctx = zdx.Context()
    m = [ctx.register_mesh(t) for t in (synth.icosphere(1), synth.box_wall(1.2, 1.1, 1.0), synth.star_mesh(4, 2))]
    rng = np.random.default_rng(3)
    pairs = []
    for a, b, d in ((0, 1, 1.1), (1, 1, 0.9), (2, 2, 1.2), (2, 0, 1.5), (0, 0, 3.0)):
        q = rng.normal(size=(2, 4))
        q /= np.linalg.norm(q, axis=1, keepdims=True)
        u = rng.normal(size=3)
        pairs.append((m[a], m[b], np.zeros(3), q[0], d * u / np.linalg.norm(u), q[1]))
    return ctx, pairs


def call(ctx, pairs, idx, **kw):
    c = [np.array([pairs[k][f] for k in idx]) for f in range(6)]
    return ctx.contact_pairs(*c, **kw)


def split(r, p):
    """The bytes of pair p."""
    lo = r["loop_offset"]
    out = [r[k][p] for k in ("tri_checks", "n_segments", "n_comps", "n_loops_raw")]
    out.append(r["loops"][lo[p]:lo[p + 1]])
    if "loop_jac" in r:
        out.append(r["loop_jac"][lo[p]:lo[p + 1]])
    if "vtx_offset" in r:
        vo = r["vtx_offset"]
        out += [np.diff(vo[lo[p]:lo[p + 1] + 1]), r["loop_vtx"][vo[lo[p]]:vo[lo[p + 1]]]]
    if "seg_offset" in r:
        out.append(r["segments"][r["seg_offset"][p]:r["seg_offset"][p + 1]])
    return b"".join(np.ascontiguousarray(x).tobytes() for x in out)


@pytest.mark.parametrize("n,kw", [
    (1, dict(segments=True)), (64, dict(segments=True, mode=zdx.MODE_PLAIN)), (65, dict(segments=True, sensitivities=True)),
    (512, dict(segments=True, noalloc=True)), (513, dict(segments=True)), (513, dict(sensitivities=True, mode=zdx.MODE_PLAIN)),
    (7001, dict(segments=True)), (66001, dict(segments=True, vertices=False)),
])
def test_pair_bytes_do_not_depend_on_the_call(base, n, kw):
    ctx, pairs = base
    one = call(ctx, pairs, range(len(pairs)), **{k: v for k, v in kw.items() if k not in ("mode", "noalloc")})
    want = [split(one, p) for p in range(len(pairs))]
    assert int(one["loop_offset"][-1]) >= 4 and int(one["n_segments"][-1]) == 0
    idx = np.arange(n) % len(pairs) if n > 1 else np.array([2])
    r = call(ctx, pairs, idx, **kw)
    for p in range(n):
        assert split(r, p) == want[idx[p]], p

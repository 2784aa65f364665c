"""GPU: wall contacts against the oracle's (area, point, normal), on meshes and
sections on either side of what the kernel holds in LDS (1280 vertices, 96
section points), with the Jacobian's flag on and off giving the same record."""
import numpy as np
import pytest

import oracle as O
from zdx import synth

zdx = pytest.importorskip("zdx")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tris", [synth.box_wall(1.0, 1.2, 0.9), synth.icosphere(2), synth.star_mesh(7, 3),
                                  synth.star_hull_mesh(5, 1280), synth.star_hull_mesh(5, 1283), synth.icosphere(4)],
                         ids=["box", "ico2", "star3", "1280", "1283", "ico4"])
def test_wall_contacts_match_oracle(tris):
    ctx = zdx.Context(0)
    mid = ctx.register_mesh(tris, center=False)
    tol = ctx.mesh_props[mid][5] * 0.1   # a tenth of the mean edge
    g = np.random.default_rng(2)
    pos = g.uniform(-0.1, 0.1, (6, 3)) + np.array([0, 0, 0.3])
    quat = g.normal(size=(6, 4))
    quat /= np.linalg.norm(quat, axis=1, keepdims=True)
    wall = np.array([[[-3, -3, 0], [3, -3, 0], [0, 4, 0]], [[-3, -3, 9], [3, -3, 9], [0, 4, 9]],
                     [[0.1, -3, 0.2], [0.2, 3, 0.2], [0.1, 0, 2.0]], [[-0.1, 0, 0.1], [0.1, 0, 0.1], [0, 0.1, 0.1]]], float)
    nrm = np.cross(wall[:, 1] - wall[:, 0], wall[:, 2] - wall[:, 0])
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    got = ctx.wall_contacts([mid] * 6, pos, quat, wall, nrm)
    jac = ctx.wall_contacts([mid] * 6, pos, quat, wall, nrm, jac=True)
    want = np.zeros((6, 4, 8))
    body = np.ascontiguousarray(tris, float).reshape(-1)
    for b in range(6):
        for w in range(4):
            a, xc, n = np.zeros(1), np.zeros(3), np.zeros(3)
            if O.lib().orc_wall_contact(body, len(tris), pos[b], quat[b], wall[w].reshape(-1), nrm[w], tol, a, xc, n):
                want[b, w, 0], want[b, w, 1], want[b, w, 2:5] = 1.0, a[0], xc
                want[b, w, 5:8] = -n if np.dot(n, pos[b] - xc) < 0.0 else n
    assert want[:, 0, 0].all() and not want[:, 1, 0].any()
    # the same arithmetic on both sides: equal, not close
    assert np.array_equal(got[..., :8], want)
    assert np.array_equal(jac[..., :8], want) and np.isfinite(jac).all()
    ctx.close()

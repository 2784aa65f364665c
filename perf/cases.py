"""Cases by which the contact step's speed is measured.

Each case is one thing a user of the framework has it do, through the public
entry points of the `zdx` package:

  contact     zdx_contact_pairs on a batch of independent mesh pairs, into
              buffers the caller holds (the per-pair tool, offline evaluation
              of many pairs)
  gradient    PairContact forward and backward (contact geometry and its
              derivatives for the poses)
  wall        Context.wall_contacts with derivatives (the wall part of the
              differentiable step)
  sim         Sim: a rollout of `steps` time steps from a given state, with
              the state, forces and counters read back at the end
  trajectory  simulate(): the differentiable rollout, forward and adjoint

listed() names the sizes measured every time, draw() gives others of the same
ranges, prepare() makes what a program has in hand before the call, run() is
one pass, work() the bytes and operations that pass cannot do without, and
exact() what plain numpy in double precision gives for it.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "zedm-x_amd"))

import zdx  # noqa: E402
from zdx import autograd as A  # noqa: E402
from zdx import synth  # noqa: E402
from zdx import workloads as W  # noqa: E402


def listed():
    return [
        # the per-pair tool on two ellipsoid hulls: one pair, every output asked for
        dict(name="contact_one", kind="contact", meshes="ellipsoid", pairs=1, batched=True, split=True, tol=0.0,
             segments=True),
        # a small ragged batch of convex hulls of 32 to 512 points, unsplit and in plain mode, with a tolerance given
        dict(name="contact_hulls_37", kind="contact", meshes="hulls", pairs=37, batched=False, split=False, tol=2e-3,
             segments=True),
        # the batched evaluation of 4096 uneven pairs: icospheres of 80-5120 triangles, concave stars of 1280
        dict(name="contact_uneven_4096", kind="contact", meshes="uneven", pairs=4096, batched=True, split=True,
             tol=0.0, segments=False),
        # contact geometry and pose gradients of an odd batch of the same shapes
        dict(name="gradient_257", kind="gradient", meshes="uneven", pairs=257),
        # wall sections and their derivatives: hulls around the floor of a closed box of 12 triangles
        dict(name="wall_61", kind="wall", bodies=61, points=128),
        # the smallest simulation: a handful of hulls on a plane, where launches and latency count
        dict(name="sim_drop_5", kind="sim", scene="drop", bodies=5, steps=100, batched=True, model="zdem"),
        # 64 hulls on a plane and against each other, the force model the calibration uses
        dict(name="sim_drop_64", kind="sim", scene="drop", bodies=64, steps=60, batched=True, model="minimal"),
        # a medium granular bed, one launch per stage (plain mode), with the normal damping switched on
        dict(name="sim_bed_5003", kind="sim", scene="bed", bodies=5003, box=0.0741, steps=20, batched=False,
             model="damped"),
        # the headline workload: the granular bed of 100k polyhedra in a 0.2 m box
        dict(name="sim_bed_100k", kind="sim", scene="bed", bodies=100_000, box=0.2, steps=50, batched=True,
             model="zdem"),
        # a dense packing of concave stars of 320-2560 triangles, three candidate pairs per particle
        dict(name="sim_packing_60k", kind="sim", scene="packing", bodies=60_000, steps=6, batched=True,
             model="zdem"),
        # gradients of a rollout for calibration: 64 hulls, forward and adjoint
        dict(name="trajectory_64", kind="trajectory", bodies=64, steps=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["contact", "contact", "gradient", "wall", "sim", "sim", "sim", "trajectory"])
    if kind == "contact":
        return dict(kind=kind, meshes=rng.choice(["hulls", "uneven"]), pairs=_log(rng, 1, 4000),
                    batched=rng.random() < 0.6, split=rng.random() < 0.7, tol=rng.choice([0.0, 0.0, 2e-3]),
                    segments=rng.random() < 0.5)
    if kind == "gradient":
        return dict(kind=kind, meshes=rng.choice(["hulls", "uneven"]), pairs=_log(rng, 1, 1000))
    if kind == "wall":
        return dict(kind=kind, bodies=_log(rng, 1, 400), points=_log(rng, 16, 512))
    if kind == "trajectory":
        return dict(kind=kind, bodies=_log(rng, 2, 100), steps=rng.randint(3, 15))
    scene = rng.choice(["drop", "bed", "packing"])
    model, batched = rng.choice(["zdem", "minimal", "damped"]), rng.random() < 0.6
    if scene == "drop":
        return dict(kind=kind, scene=scene, bodies=_log(rng, 2, 300), steps=rng.randint(20, 100), batched=batched,
                    model=model)
    if scene == "bed":
        n = _log(rng, 300, 80_000)
        return dict(kind=kind, scene=scene, bodies=n, box=round(math.ceil(n ** (1.0 / 3.0)) * 4.12e-3, 5),
                    steps=rng.randint(5, 30), batched=batched, model=model)
    return dict(kind=kind, scene=scene, bodies=_log(rng, 1000, 50_000), steps=rng.randint(2, 6), batched=batched,
                model=model)


# ------------------------------------------------------------------ inputs
def _centred(tris):
    return tris - W._centroid(tris)


def _quats(g, n):
    q = g.normal(size=(n, 4))
    return q / np.linalg.norm(q, axis=1, keepdims=True)


def _pairs(case, seed):
    """Meshes and poses of a batch: (meshes, a, b, posA, quatA, posB, quatB)."""
    n = case["pairs"]
    g = np.random.Generator(np.random.PCG64(seed))
    if case["meshes"] == "uneven":
        meshes, _, pr = W.uneven_pairs(n, seed)
        a, b = np.array([p[0] for p in pr]), np.array([p[1] for p in pr])
        return (meshes, a, b) + tuple(np.array([p[k] for p in pr], dtype=np.float64).reshape(n, -1)
                                      for k in (2, 3, 4, 5))
    if case["meshes"] == "ellipsoid":
        # end to end along the long axis, each turned about it
        meshes = [synth.ellipsoid_hull(200, (1.0, 0.6, 0.4), 1 + seed % 1000)]
        th = g.uniform(0.0, math.pi, (2, n))
        q = np.zeros((2, n, 4))
        q[..., 0], q[..., 1] = np.cos(th), np.sin(th)
        posB = np.zeros((n, 3))
        posB[:, 0] = g.uniform(1.90, 1.95, n)
        z = np.zeros(n, dtype=np.int64)
        return meshes, z, z, np.zeros((n, 3)), q[0], posB, q[1]
    # hulls: convex, 1 to 5 % of the radii deep along a random direction
    meshes = [synth.sphere_hull(m, 7 * seed % 100_003 + m) for m in (32, 64, 128, 256, 512)]
    rad = np.array([W._centred_radius(t) for t in meshes])
    a, b = g.integers(0, len(meshes), n), g.integers(0, len(meshes), n)
    d = g.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    posA = g.uniform(-1.0, 1.0, (n, 3))
    return (meshes, a, b, posA, _quats(g, n),
            posA + d * ((rad[a] + rad[b]) * (1.0 - g.uniform(0.06, 0.10, n)))[:, None], _quats(g, n))


def _drop(case, seed):
    # starts touching the plane and the neighbours: contacts from the first step
    return W.drop_on_plane(case["bodies"], seed, height=-0.3e-3, gap=-0.35e-3)


def _workload(case, seed):
    if case["scene"] == "drop":
        return _drop(case, seed)
    if case["scene"] == "bed":
        return W.granular_bed(case["bodies"], seed=seed, box=case["box"])
    n = case["bodies"]
    return W.concave_packing(n, seed=seed, box=max(0.52 * (n / 1e6) ** (1.0 / 3.0), 0.06), n_templates=8,
                             radius_levels=32)


def _wall_inputs(case, seed):
    """Hulls placed over the floor of a unit box, most of them cutting it."""
    g = np.random.Generator(np.random.PCG64(seed))
    n = case["bodies"]
    hull = 0.1 * synth.sphere_hull(case["points"], 11 * seed % 100_003 + 1)
    pos = np.stack([g.uniform(0.02, 0.98, n), g.uniform(0.02, 0.98, n), g.uniform(0.03, 0.11, n)], 1)
    tris = synth.box_wall(1.0, 1.0, 1.0) + 0.5
    nrm = np.cross(tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0])
    return hull, pos, _quats(g, n), tris, nrm / np.linalg.norm(nrm, axis=1, keepdims=True)


def _room(case):
    """Rows the caller holds for (loops, loop vertices, segments) of a batch."""
    n = case["pairs"]
    return 8 * n + 64, 96 * n + 4096, 96 * n + 4096 if case["segments"] else 0


def _call(case, a, b, poses):
    """zdx_contact_pairs' arguments: pair records, options, output buffers."""
    n = case["pairs"]
    rec = np.zeros(n, dtype=zdx.PAIR_IN_DTYPE)
    rec["mesh_a"], rec["mesh_b"] = a, b
    rec["pos_a"], rec["quat_a"], rec["pos_b"], rec["quat_b"] = poses
    opts = zdx.ContactOpts(int(case["split"]), zdx.MODE_BATCHED if case["batched"] else zdx.MODE_PLAIN, 1e6, 0, 0,
                           case["tol"])
    loops, vtx, seg = _room(case)
    i4, f8 = np.int32, np.float64
    r = dict(tri_checks=np.zeros(n, np.int64), n_segments=np.zeros(n, i4), n_comps=np.zeros(n, i4),
             n_loops_raw=np.zeros(n, i4), loop_offset=np.zeros(n + 1, i4), loop_rec=np.zeros((loops, 28), f8),
             vtx_offset=np.zeros(loops + 1, i4), loop_vtx=np.zeros((vtx, 3), f8))
    if seg:
        r["seg_offset"], r["segments"] = np.zeros(n + 1, i4), np.zeros((seg, 6), f8)
    out = zdx.PairOut(loop_cap=loops, vtx_cap=vtx, seg_cap=seg, **{k: v.ctypes.data for k, v in r.items()})
    return rec, opts, out, r


MODELS = dict(zdem=(zdx.FORCE_ZDEM, 0.0), minimal=(zdx.FORCE_MINIMAL, 1e6), damped=(zdx.FORCE_ZDEM_DAMPED, 0.0))
# steps before the measured state, in plain mode: the bed's particles start
# apart and meet within 300 steps; the others touch from the start, and their
# first steps size the buffers
SETTLE = dict(drop=20, bed=300, packing=3)


def prepare(case, seed):
    ctx = zdx.Context(0)
    s = dict(case=case, ctx=ctx)
    if case["kind"] in ("contact", "gradient"):
        meshes, a, b, pa, qa, pb, qb = _pairs(case, seed)
        ids = np.array([ctx.register_mesh(t) for t in meshes], dtype=np.int64)
        s["a"], s["b"], s["poses"] = ids[a], ids[b], (pa, qa, pb, qb)
        if case["kind"] == "contact":
            s["in"], s["opts"], s["out"], s["res"] = _call(case, s["a"], s["b"], s["poses"])
        else:
            g = torch.Generator().manual_seed(seed)
            s["poses"] = tuple(torch.from_numpy(np.ascontiguousarray(x)) for x in s["poses"])
            # the loss's gradient, as many rows as the pairs can have loops
            s["g"] = torch.randn((16 * case["pairs"], 6), generator=g, dtype=torch.float64)
    elif case["kind"] == "wall":
        hull, s["pos"], s["quat"], s["tris"], s["normals"] = _wall_inputs(case, seed)
        s["mesh"] = np.full(case["bodies"], ctx.register_mesh(hull))
    elif case["kind"] == "sim":
        wl = _workload(case, seed)
        s["sim"], _ = W.build_sim(ctx, wl)
        s["sim"].set_force_model(*MODELS[case["model"]])
        s["mode"] = zdx.MODE_BATCHED if case["batched"] else zdx.MODE_PLAIN
        s["sim"].step(SETTLE[case["scene"]], zdx.MODE_PLAIN)
        s["sim"].step(1, s["mode"])
        s["state"] = s["sim"].state()
    else:
        scene, x, q, v = A.scene_from_workload(ctx, _drop(case, seed))
        z = torch.zeros_like(x)
        s["scene"], s["start"] = scene, (x, q, v, z, z.clone())
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    case, ctx = s["case"], s["ctx"]
    if case["kind"] == "contact":
        st = zdx.lib().zdx_contact_pairs(ctx.h, s["in"].ctypes.data, case["pairs"], ctypes.byref(s["opts"]),
                                         ctypes.byref(s["out"]))
        if st != zdx.OK:
            raise zdx.ZdxError(st, zdx.lib().zdx_last_error(ctx.h).decode())
        return s["res"]
    if case["kind"] == "gradient":
        p = [x.clone().requires_grad_(True) for x in s["poses"]]
        Sc, xc, pair = A.PairContact.apply(*p, ctx, s["a"], s["b"], True)
        g = s["g"][:len(Sc)]
        torch.autograd.backward((Sc, xc), (g[:, :3], g[:, 3:]))
        geo = torch.zeros((len(s["g"]), 6), dtype=torch.float64)
        geo[:len(Sc), :3], geo[:len(Sc), 3:] = Sc.detach(), xc.detach()
        return dict(geometry=geo, grads=[x.grad for x in p])
    if case["kind"] == "wall":
        r = ctx.wall_contacts(s["mesh"], s["pos"], s["quat"], s["tris"], s["normals"], jac=True)
        return dict(contact=r[..., :8], jac=r[..., 8:])
    if case["kind"] == "sim":
        sim = s["sim"]
        sim.set_state(s["state"])
        counters = sim.step(case["steps"], s["mode"])
        F, T, contacts = sim.forces()
        return dict(state=sim.state(), F=F, T=T, contacts=contacts, counters=counters)
    p = [x.clone().requires_grad_(True) for x in s["start"]]
    k = torch.tensor(1e6, dtype=torch.float64, requires_grad=True)
    e = torch.tensor(0.5, dtype=torch.float64, requires_grad=True)
    out = A.simulate(s["scene"], k, e, *p, steps=case["steps"], ckpt_every=8)
    loss = sum((o * o).sum() for o in out)
    loss.backward()
    return dict(final=[o.detach() for o in out], grads=[x.grad for x in p], k=k.grad, e=e.grad)


# ------------------------------------------------------------------ work
def work(case):
    """One pass: poses, states and mesh tables read once, results written
    once; 60 operations per vertex moved, 24 per triangle culled, 200 per
    intersecting triangle pair."""
    if case["kind"] in ("contact", "gradient"):
        v = {"ellipsoid": 200, "hulls": 200, "uneven": 700}[case["meshes"]]   # mean vertices of a body
        sg = {"ellipsoid": 60, "hulls": 25, "uneven": 80}[case["meshes"]]     # segments of a pair
        n = case["pairs"]
        return dict(bytes=n * (112 + 8 * 28 + 24.0 * sg) + 6 * v * 48.0,
                    flops=n * (2.0 * v * 60 + 4.0 * v * 24 + 200.0 * sg * (4 if case["kind"] == "gradient" else 1)))
    if case["kind"] == "wall":
        n, m = case["bodies"], case["points"]
        return dict(bytes=n * (56 + 12 * 256.0) + 48.0 * m, flops=n * m * (60 + 12 * 6.0))
    if case["kind"] == "trajectory":
        n, t = case["bodies"], case["steps"]
        return dict(bytes=3.0 * t * n * 256, flops=3.0 * t * n * (128 * 90 + 1000.0))
    n, t = case["bodies"], case["steps"]
    # mean vertices of a body, bodies with a partner or a wall, candidate pairs per body
    v, near, prs = {"drop": (128, 1.0, 2.0), "bed": (300, 0.2, 0.12), "packing": (700, 1.0, 3.0)}[case["scene"]]
    return dict(bytes=float(t) * n * (2 * 128 + 17 * 8 + near * v * (24 + 24)),
                flops=float(t) * n * (400 + near * v * 60 + prs * (4.0 * v * 24 + 200 * 30)))


# ------------------------------------------------------------------ numpy in 64 bits
def _rot(q):
    w, x, y, z = (q / np.linalg.norm(q, axis=-1, keepdims=True)).T
    return np.stack([np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)], -1),
                     np.stack([2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)], -1),
                     np.stack([2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], -1)], -2)


def _planes(t):
    n = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    n = n / np.linalg.norm(n, axis=1, keepdims=True)
    return n, -np.einsum("ij,ij->i", n, t[:, 0])


def _inside(p, t, n):
    ok = np.ones(len(p), dtype=bool)
    for k in range(3):
        e = t[:, (k + 1) % 3] - t[:, k]
        ok &= np.einsum("ij,ij->i", np.cross(e, p - t[:, k]), n) >= -1e-10
    return ok


def _segments(TA, TB):
    """Intersection segments of two triangle soups in (ta, tb) order."""
    loA, hiA, loB, hiB = TA.min(1), TA.max(1), TB.min(1), TB.max(1)
    ia, ib = [], []
    for c in range(0, len(TA), 256):
        sl = slice(c, c + 256)
        o = np.ones((len(TA[sl]), len(TB)), dtype=bool)
        for k in range(3):
            o &= (hiA[sl, None, k] >= loB[None, :, k]) & (loA[sl, None, k] <= hiB[None, :, k])
        r = np.nonzero(o)
        ia.append(r[0] + c)
        ib.append(r[1])
    ia, ib = np.concatenate(ia), np.concatenate(ib)
    a, b = TA[ia], TB[ib]
    (nA, dA), (nB, dB) = _planes(a), _planes(b)
    tau = np.cross(nA, nB)
    lt = np.linalg.norm(tau, axis=1)
    fine = lt >= 1e-20
    tau = tau / np.where(fine, lt, 1.0)[:, None]
    pts, use = [], []
    for t, o, n, d in ((a, b, nB, dB), (b, a, nA, dA)):
        for k in range(3):
            p0, u = t[:, k], t[:, (k + 1) % 3] - t[:, k]
            den = np.einsum("ij,ij->i", n, u)
            s = -(np.einsum("ij,ij->i", n, p0) + d) / np.where(np.abs(den) < 1e-30, 1.0, den)
            ok = (np.abs(den) >= 1e-30) & (s >= -1e-10) & (s <= 1.0 + 1e-10)
            p = p0 + u * np.clip(s, 0.0, 1.0)[:, None]
            ok &= _inside(p, o, n)
            for q, w in zip(pts, use):
                ok &= ~(w & (((p - q) ** 2).sum(1) <= 1e-18))
            pts.append(p)
            use.append(ok)
    P, use = np.stack(pts, 1), np.stack(use, 1)
    t = np.einsum("ijk,ik->ij", P, tau)
    i0 = np.where(use, t, np.inf).argmin(1)
    i1 = np.where(use, t, -np.inf).argmax(1)
    r = np.arange(len(P))
    p0, p1 = P[r, i0], P[r, i1]
    keep = fine & (use.sum(1) >= 2) & (i0 != i1) & (((p1 - p0) ** 2).sum(1) >= 1e-18)
    return np.concatenate([p0, p1], 1)[keep]


def _clip(poly, tri):
    """Sutherland-Hodgman of a 2-D point list against a triangle."""
    c1 = tri[2]
    for c2 in tri:
        e = c2 - c1
        inside = [e[0] * (p[1] - c1[1]) - e[1] * (p[0] - c1[0]) >= 0.0 for p in poly]
        out = []
        for m in range(len(poly)):
            s, p = poly[m - 1], poly[m]
            if inside[m] != inside[m - 1]:
                dc, dp = c1 - c2, s - p
                n1, n2 = c1[0] * c2[1] - c1[1] * c2[0], s[0] * p[1] - s[1] * p[0]
                n3 = dc[0] * dp[1] - dc[1] * dp[0]
                out.append((n1 * dp - n2 * dc) / n3 if abs(n3) >= 1e-30 else s)
            if inside[m]:
                out.append(p)
        poly = out
        if not poly:
            break
        c1 = c2
    return poly


def _wall_record(verts, pos, tri, nrm, tol):
    """The contact record of one body (its world triangles) with one wall
    triangle: the section's points in edge order, those within tol of an
    earlier one dropped, clipped by the triangle."""
    r = np.zeros(8)
    d0 = verts @ nrm - tri[0] @ nrm
    d1 = np.roll(d0, -1, axis=1)
    hit = d0 * d1 < 0.0
    s = np.where(hit, d0 / np.where(hit, d0 - d1, 1.0), 0.0)[..., None]
    pts = []
    for p in (verts + s * (np.roll(verts, -1, axis=1) - verts))[hit]:
        if not pts or ((np.array(pts) - p) ** 2).sum(1).min() > tol * tol:
            pts.append(p)
    if len(pts) < 3:
        return r
    u = np.cross(nrm, [1.0, 0.0, 0.0] if abs(nrm[0]) < 0.9 else [0.0, 1.0, 0.0])
    u = u / np.linalg.norm(u)
    uv = np.stack([u, np.cross(nrm, u)])
    poly = _clip(list((np.array(pts) - tri[0]) @ uv.T), (tri - tri[0]) @ uv.T)
    if len(poly) < 3:
        return r
    poly = np.array(poly)
    nx = np.roll(poly, -1, axis=0)
    area = 0.5 * abs((poly[:, 0] * nx[:, 1] - poly[:, 1] * nx[:, 0]).sum())
    if area < 0.01 * tol * tol:
        return r
    xc = tri[0] + poly.mean(0) @ uv
    r[0], r[1], r[2:5], r[5:8] = 1.0, area, xc, nrm if nrm @ (pos - xc) >= 0.0 else -nrm
    return r


def exact(case, seed):
    """The intersection segments of a batch of pairs and the wall contacts.
    What follows the segments (components, snapping within a tolerance,
    loops) and the rollouts, which carry it through every step, are decisions
    rather than formulas and have no value of this kind."""
    if case["kind"] == "contact" and case["segments"] and case["pairs"] <= 200:
        meshes, a, b, pa, qa, pb, qb = _pairs(case, seed)
        cen = [_centred(t) for t in meshes]
        RA, RB = _rot(qa), _rot(qb)
        seg = [_segments(cen[a[p]] @ RA[p].T + pa[p], cen[b[p]] @ RB[p].T + pb[p]) for p in range(case["pairs"])]
        rows = np.zeros((_room(case)[2], 6))
        seg = np.concatenate(seg)
        rows[:len(seg)] = seg
        return dict(segments=rows)
    if case["kind"] == "wall" and case["bodies"] <= 200:
        hull, pos, quat, tris, nrm = _wall_inputs(case, seed)
        c = _centred(hull)
        e = np.linalg.norm(c[:, [1, 2, 0]] - c, axis=2)
        tol = 0.1 * e.mean()
        R = _rot(quat)
        rec = np.stack([[_wall_record(c @ R[i].T + pos[i], pos[i], tris[t], nrm[t], tol) for t in range(len(tris))]
                        for i in range(len(pos))])
        return dict(contact=rec, jac=None)
    return None

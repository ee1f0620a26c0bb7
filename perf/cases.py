"""What a user of this framework has it do, as cases that can be timed and compared.

Every case is one pass through the package's public entry points, on inputs made from a seed:

  rays      TriMesh.toi_and_normal_with_ray: a sensor's or renderer's rays against a terrain
  pairs     query.contact of a small batch of balls and boxes: one frame of a small game scene
  hulls     query.contact and query.distance of convex hull pairs: a batched narrow phase
  scene     World.step on two consecutive frames (a tree rebuild and a refit), with the contacts
  toi       query.time_of_impact of moving shapes: continuous collision checks
  shots     query.cast_rays of rays against chosen shapes: picking, line-of-sight
  world     World.first_interference_with_rays: rays through a whole scene
  terrain   TriMesh.contact_with_shapes and TriMesh.distance_to_shapes: objects on a terrain
  manifolds ContactManifolds: persistent contacts of a scene's pairs over two frames
  mlp       WarmStartMLP.grad: one mini-batch of the learned warm start's training

Sizes are those of the package's workloads (ncollide_amd.workloads, bench.py) and of their smaller
and odd-sized relatives.  A new scene draws its hulls from a pool of distinct hulls, as scenes that
place many copies of their models do.
"""
import math

import numpy as np
import torch

import ncollide_amd as ncx
from ncollide_amd import query, workloads
from ncollide_amd.shape import BALL, CAPSULE, CONVEX_HULL, CUBOID, SHAPE_DTYPE
from ncollide_amd.warmstart import NPARAMS, WarmStartMLP
from ncollide_amd.world import World


def listed():
    return [
        # a handful of rays against a small patch: launch latency
        {"name": "rays_small", "kind": "rays", "rays": 2048, "cells": 32, "soa": False},
        # the benchmark's batch: 1,048,576 rays, 131,072 triangles, rays kept as six arrays
        {"name": "rays_large", "kind": "rays", "rays": 1 << 20, "cells": 256, "soa": True},
        # the pairs of one frame of 1,024 balls and boxes: launch latency
        {"name": "pairs_small", "kind": "pairs", "shapes": 1024, "pairs": 283, "prediction": 0.0},
        # contact and distance of 262,144 hull pairs of 8 to 256 vertices, half of them penetrating
        {"name": "hulls_large", "kind": "hulls", "pairs": 1 << 18, "nmax": 256},
        # 1,024 balls and boxes, stepped: launch latency
        {"name": "scene_small", "kind": "scene", "shapes": 1024, "clusters": False},
        # 1,048,576 mixed shapes in clusters, stepped: the largest scene
        {"name": "scene_large", "kind": "scene", "shapes": 1 << 20, "clusters": True},
        # 262,144 mixed pairs moving toward each other
        {"name": "toi_large", "kind": "toi", "pairs": 1 << 18, "target": 0.0},
        # an odd number of rays, each against its own shape of a mixed scene
        {"name": "shots_odd", "kind": "shots", "rays": 1000003, "shapes": 1 << 18, "solid": True},
        # steep rays through a clustered scene
        {"name": "world_rays", "kind": "world", "rays": 1 << 19, "shapes": 1 << 18, "host": False},
        # mixed shapes over a terrain of 131,072 triangles: deepest contact and distance
        {"name": "terrain_shapes", "kind": "terrain", "queries": 1 << 16, "cells": 256, "prediction": 0.0},
        # persistent manifolds of the pairs of a 65,536-shape scene
        {"name": "manifolds", "kind": "manifolds", "shapes": 1 << 16},
        # a training mini-batch of the warm start's network
        {"name": "mlp_batch", "kind": "mlp", "batch": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("rays", "pairs", "hulls", "scene", "toi", "shots", "world", "terrain", "manifolds", "mlp"))
    if kind == "rays":
        return {"kind": kind, "rays": _log_int(rng, 1000, 1 << 20), "cells": _log_int(rng, 16, 256),
                "soa": rng.random() < 0.5}
    if kind == "pairs":
        n = _log_int(rng, 512, 2048)
        return {"kind": kind, "shapes": n, "pairs": int(n * rng.uniform(0.2, 0.4)), "prediction": rng.choice((0.0, 0.05))}
    if kind == "hulls":
        return {"kind": kind, "pairs": _log_int(rng, 1000, 1 << 18), "nmax": rng.choice((32, 64, 256))}
    if kind == "scene":
        return {"kind": kind, "shapes": _log_int(rng, 1000, 1 << 19), "clusters": rng.random() < 0.75}
    if kind == "toi":
        return {"kind": kind, "pairs": _log_int(rng, 1000, 1 << 18), "target": rng.choice((0.0, 0.05))}
    if kind == "shots":
        return {"kind": kind, "rays": _log_int(rng, 1000, 1 << 20), "shapes": _log_int(rng, 1000, 1 << 18),
                "solid": rng.random() < 0.5}
    if kind == "world":
        return {"kind": kind, "rays": _log_int(rng, 500, 1 << 19), "shapes": _log_int(rng, 1000, 1 << 18),
                "host": rng.random() < 0.5}
    if kind == "terrain":
        return {"kind": kind, "queries": _log_int(rng, 500, 1 << 16), "cells": _log_int(rng, 32, 256),
                "prediction": rng.choice((0.0, 0.02))}
    if kind == "manifolds":
        return {"kind": kind, "shapes": _log_int(rng, 1000, 1 << 16)}
    return {"kind": kind, "batch": _log_int(rng, 500, 8192)}


# ------------------------------------------------------------------ inputs
def _rng(case, seed):
    return np.random.default_rng([int(seed), sum(map(ord, case["kind"]))])


def _cuda(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _hull_pool(rng, n, nmax, polyhedra=False):
    """(points, offset, count) of n distinct hulls of up to nmax jittered ellipsoid points, and the
    half axes they were drawn with (polyhedra: every hull has a polyhedral structure; no axes)."""
    if polyhedra:
        return workloads.polyhedral_hulls(rng, n, 8, nmax) + (None,)
    counts = rng.integers(8, nmax + 1, n).astype(np.uint32)
    offs = np.zeros(n, np.uint32)
    offs[1:] = np.cumsum(counts)[:-1]
    axes = rng.uniform(0.2, 1.0, (n, 3))
    pts = workloads.unit_vectors(rng, int(counts.sum())) * np.repeat(axes, counts, axis=0)
    pts = (pts * (1.0 + rng.uniform(-0.02, 0.02, (len(pts), 1)))).astype(np.float32)
    return workloads.build_hulls(pts, offs, counts) + (axes,)


def _mixed(rng, n, nhulls=4096, polyhedra=False):
    """n records of balls, cuboids, capsules and hulls (8 to 64 points), one in four each."""
    pool, hoff, hcnt, _ = _hull_pool(rng, nhulls, 64, polyhedra)
    rec = np.zeros(n, SHAPE_DTYPE)
    types = rng.integers(0, 4, n).astype(np.uint32)
    p = rng.uniform(0.1, 0.5, (n, 3)).astype(np.float32)
    rec["type"] = types
    rec["p0"] = np.where(types != CONVEX_HULL, p[:, 0], 0)
    rec["p1"] = np.where(types == CUBOID, p[:, 1], np.where(types == CAPSULE, 0.05 + 0.625 * (p[:, 1] - 0.1), 0))
    rec["p2"] = np.where(types == CUBOID, p[:, 2], 0)
    pick = rng.integers(0, nhulls, n)
    rec["hull_offset"] = np.where(types == CONVEX_HULL, hoff[pick], 0)
    rec["hull_count"] = np.where(types == CONVEX_HULL, hcnt[pick], 0)
    return rec, pool


def _places(rng, n):
    """Positions in Gaussian clusters of about 16,384 shapes (sigma 5; a smaller scene is one cluster
    as dense), in a box of constant density."""
    box = 200.0 * (n / (1 << 20)) ** (1.0 / 3.0)
    centres = rng.uniform(0, box, (max(1, n >> 14), 3))
    t = centres[rng.integers(0, len(centres), n)] + rng.normal(0, 5.0 * min(1.0, n / 16384) ** (1.0 / 3.0), (n, 3))
    return np.clip(t, 0, box).astype(np.float32), box


def _balls_and_boxes(rng, n):
    """Half balls, half boxes of radius / half extents 0.1 to 0.5, 1,024 of them to a box of 20."""
    rec = np.zeros(n, SHAPE_DTYPE)
    rec["type"] = np.where(np.arange(n) < n // 2, BALL, CUBOID)
    p = rng.uniform(0.1, 0.5, (n, 3))
    rec["p0"] = p[:, 0]
    rec["p1"], rec["p2"] = (np.where(rec["type"] == CUBOID, p[:, k], 0) for k in (1, 2))
    t = rng.uniform(0.0, 20.0 * (n / 1024) ** (1.0 / 3.0), (n, 3))
    return rec, np.zeros((0, 3), np.float32), workloads.poses8(t, workloads.uniform_quats(rng, n))


def _rotate(q, v):
    """v rotated by the quaternions q (i, j, k, w)."""
    t = 2.0 * torch.linalg.cross(q[..., :3], v)
    return v + q[..., 3:4] * t + torch.linalg.cross(q[..., :3], t)


def _conj(q):
    return q * torch.tensor([-1.0, -1.0, -1.0, 1.0], dtype=q.dtype, device=q.device)


def _touching(axes_a, qa, axes_b, qb, u):
    """How far apart along u the centres of two ellipsoids are when they touch, to about 1%: the
    least of h(d) / (u . d) over directions d near and around u (h: both supports along d)."""
    n = u.shape[0]
    k = torch.arange(192, device=u.device, dtype=torch.float64) + 0.5
    z = 1.0 - 2.0 * k / 192
    r = (1.0 - z * z).sqrt()
    ph = k * math.pi * (3.0 - math.sqrt(5.0))
    d = torch.stack([r * ph.cos(), r * ph.sin(), z], 1)
    best = torch.full((n,), 1e9, dtype=torch.float64, device=u.device)
    for s in range(0, n, 16384):
        e = min(n, s + 16384)
        dd = torch.cat([u[s:e, None, :], d[None].expand(e - s, -1, -1)], 1)
        c = (dd * u[s:e, None, :]).sum(2)
        h = (_rotate(_conj(qa[s:e])[:, None], dd) * axes_a[s:e, None]).norm(dim=2)
        h = h + (_rotate(_conj(qb[s:e])[:, None], dd) * axes_b[s:e, None]).norm(dim=2)
        best[s:e] = torch.where(c > 0.05, h / c.clamp_min(0.05), 1e9).min(1).values
    return best


def _height_mesh(rng, cells):
    return workloads.heightfield_mesh(int(rng.integers(1 << 30)), cells)


def prepare(case, seed):
    rng = _rng(case, seed)
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "rays":
        pts, tri = _height_mesh(rng, case["cells"])
        o, d = workloads.heightfield_rays(int(rng.integers(1 << 30)), case["rays"], 0.1 * case["cells"])
        s.update(mesh=ncx.TriMesh(pts, tri), o=_cuda(o), d=_cuda(d), soa=None)
        if case["soa"]:
            s["soa"] = [_cuda(a[:, k]) for a in (o, d) for k in range(3)]
    elif kind == "pairs":
        rec, pool, poses = _balls_and_boxes(rng, case["shapes"])
        h = np.stack([rec["p0"], rec["p1"], rec["p2"]], 1)  # a ball's other two are zero
        rad = np.where(rec["type"] == BALL, rec["p0"], np.linalg.norm(h, axis=1))
        gap = np.abs(poses[:, None, :3] - poses[None, :, :3]).max(2) - (rad[:, None] + rad[None])
        gap[np.tril_indices(len(rec))] = np.inf
        ia, ib = np.divmod(np.sort(np.argsort(gap, axis=None)[:case["pairs"]]), len(rec))  # the nearest pairs
        s.update(shapes=ncx.ShapeSet(records=rec, pool=pool), poses=_cuda(poses), ia=_cuda(ia.astype(np.int32)),
                 ib=_cuda(ib.astype(np.int32)), prediction=case["prediction"])
    elif kind == "hulls":
        n = case["pairs"]
        pool, hoff, hcnt, axes = _hull_pool(rng, 16384, case["nmax"])
        pick = rng.integers(0, len(hoff), 2 * n)
        rec = np.zeros(2 * n, SHAPE_DTYPE)
        rec["type"] = CONVEX_HULL
        rec["hull_offset"], rec["hull_count"] = hoff[pick], hcnt[pick]
        q = workloads.uniform_quats(rng, 2 * n)
        u = workloads.unit_vectors(rng, n)
        qd, ad = _cuda(q).double(), _cuda(axes[pick])
        touch = _touching(ad[0::2], qd[0::2], ad[1::2], qd[1::2], _cuda(u)).cpu().numpy()
        gap = np.where(np.arange(n) % 2 == 0, -rng.uniform(0.0, 0.1, n), rng.uniform(0.0, 0.5, n))
        t = np.zeros((2 * n, 3))
        t[1::2] = u * np.maximum(touch + gap, 0.05)[:, None]
        s.update(shapes=ncx.ShapeSet(records=rec, pool=pool), poses=_cuda(workloads.poses8(t, q)),
                 ia=torch.arange(0, 2 * n, 2, dtype=torch.int32, device="cuda"),
                 ib=torch.arange(1, 2 * n, 2, dtype=torch.int32, device="cuda"), rec=rec, pool=pool)
    elif kind == "scene":
        n = case["shapes"]
        if case["clusters"]:
            rec, pool = _mixed(rng, n)
            poses = workloads.poses8(_places(rng, n)[0], workloads.uniform_quats(rng, n))
        else:
            rec, pool, poses = _balls_and_boxes(rng, n)
        moved = poses.copy()
        moved[:, :3] += workloads.ball_samples(rng, n, 0.5)
        shapes = ncx.ShapeSet(records=rec, pool=pool)
        world = World(shapes, margin=0.02, prediction=0.0, max_pairs=max(1 << 20, 40 * n if case["clusters"] else 0))
        s.update(world=world, frames=[_cuda(poses), _cuda(moved)], poses=_cuda(poses), contacts=None)
        for _ in range(2):  # a simulation that has run a few frames
            for f in s["frames"]:
                s["poses"].copy_(f)
                world.step(s["poses"])
                world.sync()
        cap = 24 * n  # the program's own contact list
        s["contacts"] = {k: torch.zeros((cap,) + v.shape[1:], dtype=v.dtype, device="cuda")
                         for k, v in world.results().items() if k != "epa_overflow"}
    elif kind == "toi":
        n = case["pairs"]
        rec, pool = _mixed(rng, 2 * n)
        u = workloads.unit_vectors(rng, n)
        t = rng.uniform(-50, 50, (2 * n, 3))
        t[1::2] = t[0::2] + u * rng.uniform(0.5, 3.0, (n, 1)) + rng.normal(0, 0.2, (n, 3))
        v = rng.normal(0, 0.1, (2 * n, 3))
        v[1::2] -= u * rng.uniform(0.2, 1.0, (n, 1))
        s.update(shapes=ncx.ShapeSet(records=rec, pool=pool),
                 poses=_cuda(workloads.poses8(t, workloads.uniform_quats(rng, 2 * n))), vel=_cuda(v.astype(np.float32)),
                 ia=torch.arange(0, 2 * n, 2, dtype=torch.int32, device="cuda"),
                 ib=torch.arange(1, 2 * n, 2, dtype=torch.int32, device="cuda"), target=case["target"])
    elif kind == "shots":
        n, m = case["rays"], case["shapes"]
        rec, pool = _mixed(rng, m, nhulls=256)
        t, _ = _places(rng, m)
        idx = rng.integers(0, m, n).astype(np.int32)
        o = (t[idx] + rng.normal(0, 2.0, (n, 3))).astype(np.float32)
        d = (t[idx] + rng.uniform(-0.2, 0.2, (n, 3)) - o).astype(np.float32)
        s.update(shapes=ncx.ShapeSet(records=rec, pool=pool),
                 poses=_cuda(workloads.poses8(t, workloads.uniform_quats(rng, m))), idx=_cuda(idx), o=_cuda(o),
                 d=_cuda(d), solid=case["solid"], rec=rec, pool=pool)
    elif kind == "world":
        n, m = case["rays"], case["shapes"]
        rec, pool = _mixed(rng, m)
        t, box = _places(rng, m)
        poses = _cuda(workloads.poses8(t, workloads.uniform_quats(rng, m)))
        o = rng.uniform(0, box, (n, 3)).astype(np.float32)
        o[:, 2] = box + 10.0
        d = np.tile(np.array([[0.05, 0.02, -1.0]]), (n, 1)) + rng.normal(0, 0.02, (n, 3))
        world = World(ncx.ShapeSet(records=rec, pool=pool), margin=0.02, prediction=0.0, max_pairs=max(1 << 20, 40 * m))
        world.set_contacts(False)
        world.step(poses, use_graph=False)
        world.sync()
        o, d = (a.astype(np.float32) if case["host"] else _cuda(a.astype(np.float32)) for a in (o, d))
        s.update(world=world, poses=poses, o=o, d=d)
    elif kind == "terrain":
        n = case["queries"]
        pts, tri = _height_mesh(rng, case["cells"])
        rec, pool = _mixed(rng, n)
        side = 0.1 * case["cells"]
        t = np.stack([rng.uniform(0.02, 0.98, n) * side, rng.uniform(0.02, 0.98, n) * side, rng.uniform(-0.6, 1.2, n)], 1)
        s.update(mesh=ncx.TriMesh(pts, tri), shapes=ncx.ShapeSet(records=rec, pool=pool),
                 poses=_cuda(workloads.poses8(t, workloads.uniform_quats(rng, n))),
                 idx=torch.arange(n, dtype=torch.int32, device="cuda"), prediction=case["prediction"])
    elif kind == "manifolds":
        n = case["shapes"]
        rec, pool = _mixed(rng, n, nhulls=1024, polyhedra=True)
        poses = workloads.poses8(_places(rng, n)[0], workloads.uniform_quats(rng, n))
        moved = poses.copy()
        moved[:, :3] += workloads.ball_samples(rng, n, 0.025)
        shapes = ncx.ShapeSet(records=rec, pool=pool)
        world = World(shapes, margin=0.02, prediction=0.0, max_pairs=max(1 << 20, 40 * n))
        world.set_contacts(False)
        world.step(_cuda(poses), use_graph=False)
        r = world.results()
        key = torch.sort(r["ia"].long() << 32 | r["ib"].long()).values
        npairs = 4 * n  # of about 10 a shape
        key = key[torch.arange(npairs, device="cuda") * key.numel() // npairs]
        s.update(shapes=shapes, frames=[_cuda(poses), _cuda(moved)], ia=(key >> 32).int(),
                 ib=(key & 0xFFFFFFFF).int(), slots=torch.arange(npairs, dtype=torch.int32, device="cuda"),
                 state=ncx.ContactManifolds(shapes.ctx, npairs))
    elif kind == "mlp":
        n = case["batch"]
        g = torch.Generator(device="cuda").manual_seed(int(rng.integers(1 << 40)))
        mlp = WarmStartMLP(ncx.default_context())
        mlp.set_params(_weights(rng))
        x = torch.randn(n, 48, generator=g, device="cuda") * 0.6
        x[:, 44:] = 0
        y = torch.randn(n, 3, generator=g, device="cuda")
        s.update(mlp=mlp, x=x.half(), y=y / y.norm(dim=1, keepdim=True))
    return s


def _weights(rng):
    """A flat parameter vector: W1 (64 x 48), b1, W2 (64 x 64), b2, W3 (16 x 64), b3; padding zero."""
    w1, w2, w3 = rng.normal(0, 0.2, (64, 48)), rng.normal(0, 0.18, (64, 64)), rng.normal(0, 0.18, (16, 64))
    b1, b2, b3 = rng.normal(0, 0.05, 64), rng.normal(0, 0.05, 64), rng.normal(0, 0.05, 16)
    w1[:, 44:], w3[3:], b3[3:] = 0, 0, 0
    p = np.concatenate([a.ravel() for a in (w1, b1, w2, b2, w3, b3)]).astype(np.float32)
    assert p.size == NPARAMS
    return p


# ------------------------------------------------------------------ one pass
def run(s):
    kind = s["kind"]
    if kind == "rays":
        return s["mesh"].toi_and_normal_with_ray(s["o"], s["d"], 100.0, soa=s["soa"])
    if kind == "pairs":
        return query.contact(s["shapes"], s["poses"], s["ia"], s["ib"], s["prediction"])
    if kind == "hulls":
        return {"contact": query.contact(s["shapes"], s["poses"], s["ia"], s["ib"], 0.0),
                "distance": query.distance(s["shapes"], s["poses"], s["ia"], s["ib"])}
    if kind == "scene":
        for f in s["frames"]:
            s["poses"].copy_(f)
            s["world"].step(s["poses"])
        r = s["world"].results()
        for k, v in s["contacts"].items():
            v[:len(r[k])].copy_(r[k][:len(v)])
        return s["contacts"], len(r["ia"])
    if kind == "toi":
        return query.time_of_impact(s["shapes"], s["poses"], s["vel"], s["ia"], s["ib"], 10.0, s["target"])
    if kind == "shots":
        return query.cast_rays(s["shapes"], s["poses"], s["idx"], s["o"], s["d"], 50.0, s["solid"])
    if kind == "world":
        return s["world"].first_interference_with_rays(s["poses"], s["o"], s["d"], 1000.0)
    if kind == "terrain":
        return {"contact": s["mesh"].contact_with_shapes(s["shapes"], s["poses"], s["idx"], s["prediction"]),
                "distance": s["mesh"].distance_to_shapes(s["shapes"], s["poses"], s["idx"])}
    if kind == "manifolds":
        s["state"].reset(s["slots"])  # interactions that start in the first frame and persist in the second
        out = [s["state"].update(s["shapes"], f, s["ia"], s["ib"], s["slots"], 0.02, 0.05, 0.05) for f in s["frames"]]
        return {"first": out[0], "second": out[1], "dirs": s["state"].dirs(s["slots"])}
    return s["mlp"].grad(s["x"], s["y"])


def work(case):
    """Inputs read once and outputs written once; flops: the least arithmetic of the path's steps
    (a box test 12, a support scan 5 per vertex, a closed-form or simplex step about 100)."""
    kind = case["kind"]
    if kind == "rays":
        n, tri = case["rays"], 2 * case["cells"] ** 2
        return {"bytes": n * 44 + tri * 48, "flops": n * 12 * math.log2(tri)}
    if kind == "pairs":
        n = case["pairs"]
        return {"bytes": case["shapes"] * 64 + n * 57, "flops": n * 400}
    if kind == "hulls":
        n, v = case["pairs"], 0.5 * (8 + case["nmax"])
        return {"bytes": n * (8 + 128 + 53 + 8) + min(2 * n, 16384) * v * 12, "flops": n * 2 * (8 * 10 * v + 800)}
    if kind == "scene":
        n = case["shapes"]
        p = 10 * n if case["clusters"] else 0.3 * n
        return {"bytes": 2 * (n * (64 + 24 * 2) + p * 60), "flops": 2 * (n * 12 * math.log2(n) + p * 400)}
    if kind == "toi":
        return {"bytes": case["pairs"] * (8 + 152 + 54) + 4096 * 36 * 12, "flops": case["pairs"] * 1200}
    if kind == "shots":
        return {"bytes": case["rays"] * 48 + case["shapes"] * 64, "flops": case["rays"] * 600}
    if kind == "world":
        return {"bytes": case["rays"] * 44 + case["shapes"] * 88, "flops": case["rays"] * 24 * math.log2(case["shapes"])}
    if kind == "terrain":
        n = case["queries"]
        return {"bytes": n * (64 + 53) + 2 * case["cells"] ** 2 * 48, "flops": n * 20000}
    if kind == "manifolds":
        n = 4 * case["shapes"]
        return {"bytes": 2 * (n * (12 + 2 * 56 + 4 + 56) + case["shapes"] * 64), "flops": 2 * n * 600}
    return {"bytes": case["batch"] * (96 + 12) + 2 * NPARAMS * 4, "flops": case["batch"] * (14208 + 28416)}


def tolerance(case):
    if case["kind"] == "mlp":
        # 16-bit operands and activations, 32-bit sums: 7e-4 to 3e-3 from the 64-bit gradient
        return {"rel": 4e-3, "max": 0.05}
    # every query restates a reference's 32-bit operations one by one, in a fixed order, per pair or
    # ray: results are defined to the last bit and do not depend on how the work is split
    return "exact"


# ------------------------------------------------------------------ in 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind not in ("rays", "pairs", "hulls", "shots", "mlp"):
        # scene, terrain, manifolds, toi and world: exact penetration depths, times of impact and
        # nearest triangles of millions of curved or many-faced pairs take minutes in plain torch
        return None
    s = prepare(case, seed)
    if kind == "rays":
        pts, _ = _height_mesh(_rng(case, seed), case["cells"])
        return _exact_height_rays(torch.as_tensor(pts, device="cuda").double(), case["cells"], s["o"], s["d"])
    if kind == "pairs":
        # with a prediction, separated boxes have a distance for a depth, which the axes do not give
        return _exact_pairs(case, seed, s) if case["prediction"] == 0.0 else None
    if kind == "hulls":
        d = _exact_hull_distance(s["rec"], s["pool"], s["poses"])
        c = {k: None for k in ("has_contact", "world1", "world2", "normal", "depth", "gjk_iters")}
        return {"contact": c, "distance": (d, None)}
    if kind == "shots":
        return _exact_shots(s), None, None
    return _exact_mlp(_weights_of(case, seed), s["x"], s["y"])


def _weights_of(case, seed):
    rng = _rng(case, seed)
    rng.integers(1 << 40)
    return _weights(rng)


def _exact_mlp(p, x, y):
    sizes = ((64, 48), (64,), (64, 64), (64,), (16, 64), (16,))
    w, at = [], 0
    p = torch.as_tensor(p, device="cuda").double()
    for sh in sizes:
        k = math.prod(sh)
        w.append(p[at:at + k].reshape(sh).clone().requires_grad_())
        at += k
    h = torch.relu(x.double() @ w[0].T + w[1])
    h = torch.relu(h @ w[2].T + w[3])
    f = (h @ w[4].T + w[5])[:, :3]
    loss = (f - y.double()).square().sum(1).mean()
    loss.backward()
    g = [a.grad.clone() for a in w]
    g[0][:, 44:] = 0
    return torch.cat([a.reshape(-1) for a in g]), loss.detach().reshape(1)


def _exact_height_rays(pts, cells, o, d):
    """Rays walked through the height field's cells, both triangles of each cell tested."""
    nv = cells + 1
    o, d = o.double(), d.double()
    n = o.shape[0]
    size = 0.1
    dead = torch.full((n,), 1e30, dtype=torch.float64, device=o.device)
    inv = torch.where(d[:, :2].abs() > 1e-300, 1.0 / d[:, :2], 1e300)
    cell = (o[:, :2] / size).floor().long()
    cell = cell.clamp(0, cells - 1)
    step = torch.where(d[:, :2] >= 0, 1, -1)
    best, nrm = dead.clone(), torch.zeros_like(o)
    zlo = pts[:, 2].min() - 1e-6
    alive = torch.arange(n, device=o.device)
    for _ in range(2 * cells + 2):
        if not alive.numel():
            break
        oo, dd, c = o[alive], d[alive], cell[alive]
        p00 = c[:, 1] * nv + c[:, 0]
        ids = (p00, p00 + 1, p00 + nv, p00 + nv + 1)
        for i, j, l in ((0, 1, 2), (1, 3, 2)):
            a, b, e = pts[ids[i]], pts[ids[j]], pts[ids[l]]
            m = torch.linalg.cross(b - a, e - a)
            den = (m * dd).sum(1)
            t = (m * (a - oo)).sum(1) / torch.where(den != 0, den, 1.0)
            x = oo + dd * t[:, None]
            inside = (den != 0) & (t >= 0) & (t <= 100.0)
            for v, w in ((a, b), (b, e), (e, a)):
                inside &= (torch.linalg.cross(w - v, x - v) * m).sum(1) >= 0
            better = inside & (t < best[alive])
            at = alive[better]
            best[at] = t[better]
            m = m / m.norm(dim=1, keepdim=True)
            nrm[at] = torch.where(den[:, None] < 0, m, -m)[better]
        edge = (c + (step[alive] > 0).long()).double() * size
        tx = (edge - oo[:, :2]) * inv[alive]
        ax = (tx[:, 1] < tx[:, 0]).long()
        row = torch.arange(alive.numel(), device=o.device)
        leave = tx[row, ax]
        c[row, ax] += step[alive][row, ax]
        cell[alive] = c
        go = (c >= 0).all(1) & (c < cells).all(1) & (best[alive] > leave) & (oo[:, 2] + dd[:, 2] * leave >= zlo)
        alive = alive[go]
    hit = best < 1e30
    return torch.where(hit, best, -1.0), torch.where(hit[:, None], nrm, 0.0), None


def _exact_pairs(case, seed, s):
    """Depths of ball and box pairs: closed forms, and separating axes for two boxes."""
    rec, _, poses = _balls_and_boxes(_rng(case, seed), case["shapes"])
    p = torch.as_tensor(poses, device="cuda").double()
    h = torch.as_tensor(np.stack([rec["p0"], rec["p1"], rec["p2"]], 1), device="cuda").double()
    ball = torch.as_tensor((rec["type"] == BALL), device="cuda")
    ia, ib = s["ia"].long(), s["ib"].long()
    swap = ball[ib] & ~ball[ia]
    ia, ib = torch.where(swap, ib, ia), torch.where(swap, ia, ib)  # the ball first
    t = p[ib, :3] - p[ia, :3]
    bb = h[ia, 0] + h[ib, 0] - t.norm(dim=1)
    local = _rotate(_conj(p[ib, 4:]), -t)  # the ball's centre in the box's frame
    out = (local.abs() - h[ib]).clamp_min(0).norm(dim=1)
    into = (h[ib] - local.abs()).min(1).values
    bc = torch.where(out > 0, h[ia, 0] - out, h[ia, 0] + into)
    eye = torch.eye(3, dtype=torch.float64, device="cuda")
    A = torch.stack([_rotate(p[ia, 4:], eye[k].expand_as(t)) for k in range(3)], 1)
    B = torch.stack([_rotate(p[ib, 4:], eye[k].expand_as(t)) for k in range(3)], 1)
    axes = torch.cat([A, B] + [torch.linalg.cross(A[:, i], B[:, j])[:, None] for i in range(3) for j in range(3)], 1)
    ln = axes.norm(dim=2, keepdim=True)
    axes = axes / ln.clamp_min(1e-9)
    r = ((A[:, None] * axes[:, :, None]).sum(3).abs() * h[ia][:, None]).sum(2)
    r = r + ((B[:, None] * axes[:, :, None]).sum(3).abs() * h[ib][:, None]).sum(2)
    cc = (r - (axes * t[:, None]).sum(2).abs() + torch.where(ln[..., 0] < 1e-6, 1e9, 0.0)).min(1).values
    depth = torch.where(ball[ia] & ball[ib], bb, torch.where(ball[ia], bc, cc))
    depth = torch.where(depth > 0, depth, 0.0)
    return {"has_contact": None, "world1": None, "world2": None, "normal": None, "depth": depth, "gjk_iters": None}


_SUBSETS = [[i for i in range(4) if m >> i & 1] for m in range(1, 16)]


def _nearest(w):
    """The point of the hull of four points (n, 4, 3) nearest to the origin, and which of them span it."""
    n = w.shape[0]
    best = torch.full((n,), math.inf, dtype=w.dtype, device=w.device)
    point, keep = torch.zeros(n, 3, dtype=w.dtype, device=w.device), torch.zeros(n, 4, dtype=torch.bool, device=w.device)
    for sub in _SUBSETS:
        a = w[:, sub[0]]
        e = torch.stack([w[:, k] - a for k in sub[1:]], 2) if len(sub) > 1 else None
        if e is None:
            lam = torch.ones(n, 1, dtype=w.dtype, device=w.device)
            ok = torch.ones(n, dtype=torch.bool, device=w.device)
        else:
            g = e.transpose(1, 2).contiguous() @ e
            rhs = -(e * a[:, :, None]).sum(1)
            dg = torch.diagonal(g, dim1=1, dim2=2)
            ok = torch.linalg.det(g) > 1e-14 * dg.prod(1)
            g = torch.where(ok[:, None, None], g, torch.eye(len(sub) - 1, dtype=w.dtype, device=w.device))
            mu = torch.linalg.solve(g, rhs)
            lam = torch.cat([1 - mu.sum(1, keepdim=True), mu], 1)
            ok &= (lam >= 0).all(1)
        x = (w[:, sub] * lam[:, :, None]).sum(1)
        d = x.square().sum(1)
        if len(sub) == 4:
            d = torch.zeros_like(d)
        better = ok & (d < best)
        best = torch.where(better, d, best)
        point[better] = x[better] if len(sub) < 4 else 0
        row = torch.zeros(4, dtype=torch.bool, device=w.device)
        row[sub] = True
        keep[better] = row
    return point, keep


def _exact_hull_distance(rec, pool, poses):
    """Distances of the hull pairs (2k, 2k + 1): GJK in 64 bits, run to its fixed point."""
    dev = poses.device
    off, cnt = (torch.as_tensor(rec[k].astype(np.int64), device=dev) for k in ("hull_offset", "hull_count"))
    pool = torch.as_tensor(pool, device=dev).double()
    poses = poses.double()
    out = torch.zeros(len(rec) // 2, dtype=torch.float64, device=dev)
    for s in range(0, out.numel(), 65536):
        e = min(out.numel(), s + 65536)
        verts, number = [], torch.arange(s, e, device=dev)
        for side in (0, 1):
            k = 2 * number + side
            m = int(cnt[k].max())
            ids = off[k][:, None] + torch.minimum(torch.arange(m, device=dev)[None], cnt[k][:, None] - 1)
            verts.append(_rotate(poses[k, None, 4:], pool[ids]) + poses[k, None, :3])

        def support(v, live):
            a, b = verts[0][live], verts[1][live]
            i = (a * -v[:, None]).sum(2).argmax(1)
            j = (b * v[:, None]).sum(2).argmax(1)
            r = torch.arange(a.shape[0], device=dev)
            return a[r, i] - b[r, j]

        live = torch.arange(e - s, device=dev)
        v = poses[2 * number, :3] - poses[2 * number + 1, :3]
        w = support(v, live)[:, None].expand(-1, 4, -1).contiguous()
        v = w[:, 0].clone()
        for _ in range(64):
            new = support(v, live)
            vv = v.square().sum(1)
            go = (vv > 1e-20) & (vv - (v * new).sum(1) > 1e-13 * vv)
            out[s + live] = torch.where(vv > 1e-20, vv.sqrt(), 0.0)
            live, w, new, keep = live[go], w[go], new[go], (None if _ == 0 else keep[go])
            if not live.numel():
                break
            if keep is None:
                w = torch.cat([w[:, :1], new[:, None].expand(-1, 3, -1)], 1)
            else:
                first = w[torch.arange(live.numel(), device=dev), keep.long().argmax(1)]
                w = torch.where(keep[:, :, None], w, first[:, None])
                free = (~keep).long().argmax(1)
                full = keep.all(1)
                w[torch.arange(live.numel(), device=dev), free] = torch.where(full[:, None], w[:, 0], new)
            v, keep = _nearest(w)
    return out


def _exact_shots(s):
    """Entry (or, from inside a shape that is not solid, exit) parameters of the rays."""
    rec, dev = s["rec"], s["o"].device
    idx = s["idx"].long()
    p = s["poses"].double()[idx]
    o, d = s["o"].double() - p[:, :3], s["d"].double()
    o, d = _rotate(_conj(p[:, 4:]), o), _rotate(_conj(p[:, 4:]), d)
    kind = torch.as_tensor(rec["type"].astype(np.int64), device=dev)[idx]
    h = torch.as_tensor(np.stack([rec["p0"], rec["p1"], rec["p2"]], 1), device=dev).double()[idx]
    inf = torch.full_like(o[:, 0], math.inf)

    def sphere(c, r):  # entry and exit of a ball, empty as (inf, -inf)
        q = o - c
        a, b, cc = (d * d).sum(1), (q * d).sum(1), (q * q).sum(1) - r * r
        disc = b * b - a * cc
        root = disc.clamp_min(0).sqrt()
        return torch.where(disc >= 0, (-b - root) / a, inf), torch.where(disc >= 0, (-b + root) / a, -inf)

    lo, hi = sphere(torch.zeros(3, dtype=torch.float64, device=dev), h[:, 0])
    t1, t2 = (-h - o) / d, (h - o) / d
    box = torch.minimum(t1, t2).amax(1), torch.maximum(t1, t2).amin(1)
    lo, hi = torch.where(kind == CUBOID, box[0], lo), torch.where(kind == CUBOID, box[1], hi)
    up = torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64, device=dev)
    a, b, c = d[:, 0] ** 2 + d[:, 2] ** 2, o[:, 0] * d[:, 0] + o[:, 2] * d[:, 2], o[:, 0] ** 2 + o[:, 2] ** 2 - h[:, 1] ** 2
    disc = b * b - a * c
    root = disc.clamp_min(0).sqrt()
    y1, y2 = (-h[:, 0] - o[:, 1]) / d[:, 1], (h[:, 0] - o[:, 1]) / d[:, 1]
    clo = torch.maximum((-b - root) / a, torch.minimum(y1, y2))
    chi = torch.minimum((-b + root) / a, torch.maximum(y1, y2))
    empty = (disc < 0) | (clo > chi)
    parts = [sphere(up * h[:, :1], h[:, 1]), sphere(-up * h[:, :1], h[:, 1]),
             (torch.where(empty, inf, clo), torch.where(empty, -inf, chi))]
    cap = kind == CAPSULE
    lo = torch.where(cap, torch.stack([q[0] for q in parts]).amin(0), lo)
    hi = torch.where(cap, torch.stack([q[1] for q in parts]).amax(0), hi)
    # hulls: the planes through three vertices that have every vertex on one side
    off, cnt = (rec[k].astype(np.int64) for k in ("hull_offset", "hull_count"))
    isHull = rec["type"] == CONVEX_HULL
    first = torch.as_tensor(off, device=dev)[idx]
    lo, hi = lo.clone(), hi.clone()
    of_hull = torch.nonzero(kind == CONVEX_HULL).reshape(-1)
    of_hull = of_hull[torch.argsort(first[of_hull], stable=True)]
    starts, amounts = torch.unique_consecutive(first[of_hull], return_counts=True)
    count_at = dict(zip(off[isHull].tolist(), cnt[isHull].tolist()))
    at = 0
    for start, k in zip(starts.tolist(), amounts.tolist()):
        rays = of_hull[at:at + k]
        at += k
        v = torch.as_tensor(s["pool"][start:start + count_at[start]], device=dev).double()
        tri = torch.combinations(torch.arange(len(v), device=dev), 3)
        m = torch.linalg.cross(v[tri[:, 1]] - v[tri[:, 0]], v[tri[:, 2]] - v[tri[:, 0]])
        m = m / m.norm(dim=1, keepdim=True).clamp_min(1e-30)
        side = m @ v.T - (m * v[tri[:, 0]]).sum(1, keepdim=True)
        out, back = (side <= 1e-12).all(1), (side >= -1e-12).all(1)
        m = torch.cat([m[out], -m[back]])
        c = torch.cat([(m[:out.sum()] * v[tri[out, 0]]).sum(1), (m[out.sum():] * v[tri[back, 0]]).sum(1)])
        den, num = d[rays] @ m.T, c - o[rays] @ m.T
        t = num / den
        lo[rays] = torch.where(den < 0, t, -math.inf).amax(1)
        hi[rays] = torch.where(den > 0, t, math.inf).amin(1)
    hit = (lo <= hi) & (hi >= 0)
    t = torch.where(lo >= 0, lo, 0.0 if s["solid"] else hi)
    return torch.where(hit & (t <= 50.0), t, -1.0)

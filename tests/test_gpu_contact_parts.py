"""Contacts of more pairs than one part's EPA records (2^26): batches and scenes go over their pairs in
parts, and the runs that outgrow every LDS arena in one of them are made again at the end.  Every
result has the bits that the same pair has in a batch of one part."""
import numpy as np
import pytest
import torch

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from ncollide_amd.world import World
from tests.test_gpu_parity import _curved_pairs, oracle_shapes

pytestmark = pytest.mark.gpu

PART = 1 << 26
KEYS = ("has_contact", "world1", "world2", "normal", "depth", "gjk_iters")


def test_batch_of_two_parts(ctx, orc):
    n = 400000
    rec, poses8, rng = _curved_pairs(12, n)
    pool = np.zeros((1, 3), np.float32)
    ia = np.arange(0, 2 * n, 2, dtype=np.uint32)
    it = orc.contact(oracle_shapes(orc, rec, pool), to_oracle_poses(poses8), ia, ia + 1, 0.0, nthreads=8)["epa_iters"]
    longest = np.argsort(it)[-100:]  # up to 2,142 iterations: past the largest LDS arena
    assert it[longest[-1]] > 2000
    short = rng.choice(np.nonzero(it < 30)[0], 5000, replace=False)
    sel = np.concatenate([short, longest])
    idx = rng.integers(0, len(short), PART + 200001)
    idx[rng.choice(len(idx), 5000, replace=False)] = len(short) + rng.integers(0, 100, 5000)
    idx[rng.choice(len(idx), 60, replace=False)] = len(sel) - 1
    ss = ncx.ShapeSet(records=rec, pool=pool, ctx=ctx)
    poses = torch.as_tensor(poses8, device=ctx.device)
    a = torch.as_tensor(ia[sel].astype(np.int32), device=ctx.device)
    ref = ncx.query.contact(ss, poses, a, a + 1, 0.0)
    k = torch.as_tensor(idx, device=ctx.device)
    g = ncx.query.contact(ss, poses, a[k], a[k] + 1, 0.0)
    for key in KEYS:
        assert torch.equal(g[key], ref[key][k]), key


def test_scene_of_two_parts(ctx):
    n = 400000
    rng = np.random.default_rng(4)
    w = workloads.full_pipeline(seed=4, n=n // 100, box=8.0, nclusters=1, hull_nmax=16)
    rec = np.tile(w["records"], 100)
    hulls = np.nonzero(rec["type"] == workloads.CONVEX_HULL)[0]
    rec["type"][hulls[::2]] = workloads.CUBOID
    for p in ("p0", "p1", "p2"):
        rec[p][hulls[::2]] = 0.3
    t = rng.uniform(0, 15.0, (n, 3))
    poses = torch.as_tensor(workloads.poses8(t, workloads.uniform_quats(rng, n)).astype(np.float32), device=ctx.device)
    ss = ncx.ShapeSet(records=rec, pool=w["pool"], ctx=ctx)
    world = World(ss, margin=0.01, prediction=0.0, max_pairs=2 * PART)
    for step in range(4):  # the first step is not captured
        world.step(poses)
        r = world.results()
        assert PART < r["ia"].numel() < 2 * PART
        for lo in (0, PART // 2, PART):
            c = slice(lo, min(lo + PART // 2, r["ia"].numel()))
            g = ncx.query.contact(ss, poses, r["ia"][c], r["ib"][c], 0.0)
            for key in KEYS:
                assert torch.equal(g[key], r[key][c]), (step, lo, key)
        assert r["has_contact"].any() and not r["has_contact"].all()
        poses[:, :3] += torch.as_tensor(rng.normal(0, 0.005, (n, 3)).astype(np.float32), device=ctx.device)

"""Distances with one pair a lane (the scans of hulls shared by 8 lanes): batches around the smallest
that take it (32,768 pairs), and smaller ones, around a wavefront and the partition's smallest, which
take 8 lanes a pair in its place; hulls of 4 to 256 vertices next to every other shape, with and
without a warm start under an iteration cap, against the oracle and the kernel with 8 lanes a pair."""
import numpy as np
import pytest
import torch

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from tests.test_gpu_parity import oracle_shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npairs,warm", [(1, False), (63, True), (65, False), (16384, True), (16384 + 63, False),
                                         (32768, True), (32768 + 63, False)])
def test_distance_one_pair_a_lane(ctx, orc, npairs, warm):
    w = workloads.full_pipeline(seed=61, n=4000, box=12.0, nclusters=2)
    rng = np.random.default_rng(npairs)
    rec = w["records"].copy()
    verts = rng.normal(size=(4000, 3)).astype(np.float32)  # point sets; support maps need no hull of them
    hulls = np.nonzero(rec["type"] == 3)[0]
    cnt = rng.choice([4, 7, 8, 9, 31, 33, 64, 96, 97, 255, 256], len(hulls))
    rec["hull_offset"][hulls] = rng.integers(0, len(verts) - 256, len(hulls))
    rec["hull_count"][hulls] = cnt
    ia = rng.integers(0, len(rec), npairs).astype(np.uint32)
    ib = ((ia + 1 + rng.integers(0, len(rec) - 1, npairs)) % len(rec)).astype(np.uint32)
    poses = torch.as_tensor(w["poses"], device=ctx.device)
    kw = {}
    if warm:
        d0 = rng.normal(size=(npairs, 3)).astype(np.float32)
        d0[::3] = 0
        kw = {"init_dir": torch.as_tensor(d0, device=ctx.device), "max_iter": 4}
    out = []
    for variant in (0, 4):
        ss = ncx.ShapeSet(records=rec, pool=verts, ctx=ctx)
        ss.set_tuning([variant] * 4, query="distance")
        d, it = ncx.query.distance(ss, poses, ia, ib, **kw)
        out.append((d.cpu().numpy().view(np.uint32), it.cpu().numpy()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    if not warm:
        m = min(npairs, 3000)
        rd, rit = orc.distance(oracle_shapes(orc, rec, verts), to_oracle_poses(w["poses"]), ia[:m], ib[:m], nthreads=8)
        assert np.array_equal(out[1][0][:m], np.asarray(rd, np.float32).view(np.uint32))
        assert np.array_equal(out[1][1][:m], np.asarray(rit))


@pytest.mark.parametrize("nlarge", [1, 63, 65])
def test_few_pairs_of_a_bucket(ctx, orc, nlarge):
    """A batch large enough for one pair a lane (32,768 pairs) with hulls of more than 96 vertices in
    nlarge of them: the bucket's launch has less than a wavefront's pairs, or one more."""
    w = workloads.full_pipeline(seed=61, n=4000, box=12.0, nclusters=2)
    rng = np.random.default_rng(nlarge)
    rec = w["records"].copy()
    verts = rng.normal(size=(4000, 3)).astype(np.float32)
    hulls = np.nonzero(rec["type"] == 3)[0]
    rec["hull_offset"][hulls] = rng.integers(0, len(verts) - 256, len(hulls))
    rec["hull_count"][hulls] = rng.choice([4, 9, 33, 96], len(hulls))
    rec["hull_count"][hulls[0]] = 256
    others = np.delete(np.arange(len(rec)), hulls[0])
    ia, ib = rng.choice(others, (2, 32768 + 1)).astype(np.uint32)
    ia[rng.choice(len(ia), nlarge, replace=False)] = hulls[0]
    ss = ncx.ShapeSet(records=rec, pool=verts, ctx=ctx)
    ss.set_tuning([0, 3, 0, 4], query="distance")
    d, it = ncx.query.distance(ss, torch.as_tensor(w["poses"], device=ctx.device), ia, ib)
    rd, rit = orc.distance(oracle_shapes(orc, rec, verts), to_oracle_poses(w["poses"]), ia, ib, nthreads=8)
    assert np.array_equal(d.cpu().numpy().view(np.uint32), np.asarray(rd, np.float32).view(np.uint32))
    assert np.array_equal(it.cpu().numpy(), np.asarray(rit))


def test_small_batches_of_a_tuned_set(ctx):
    """One pair a lane leaves the chip idle on a few hundred pairs (186 us for 300 pairs of these hulls,
    65 us with 8 lanes a pair): a set tuned to it takes 8 lanes for them."""
    import time
    rng = np.random.default_rng(5)
    rec = np.zeros(2000, ncx.shape.SHAPE_DTYPE)
    rec["type"] = 3
    verts = rng.normal(size=(8000, 3)).astype(np.float32)
    rec["hull_offset"] = rng.integers(0, 8000 - 256, 2000)
    rec["hull_count"] = 256
    poses = torch.as_tensor(workloads.poses8(rng.uniform(0, 40, (2000, 3)), workloads.uniform_quats(rng, 2000)),
                            device=ctx.device)
    ia, ib = (torch.as_tensor(rng.integers(0, 2000, 300).astype(np.int32), device=ctx.device) for _ in range(2))
    best = {}
    for variant in (0, 4):
        ss = ncx.ShapeSet(records=rec, pool=verts, ctx=ctx)
        ss.set_tuning([variant] * 4, query="distance")
        best[variant] = np.inf
        for _ in range(60):
            torch.cuda.synchronize()
            t = time.perf_counter()
            ncx.query.distance(ss, poses, ia, ib)
            torch.cuda.synchronize()
            best[variant] = min(best[variant], time.perf_counter() - t)
    assert best[4] < 1.7 * best[0]


def test_distance_bad_index_is_refused(ctx):
    w = workloads.full_pipeline(seed=61, n=200, box=8.0, nclusters=1)
    ss = ncx.ShapeSet(records=w["records"], pool=w["pool"], ctx=ctx)
    ss.set_tuning([4] * 4, query="distance")
    poses = torch.as_tensor(w["poses"], device=ctx.device)
    ia = np.zeros(20000, np.uint32)
    ib = np.ones(20000, np.uint32)
    ib[777] = 200
    with pytest.raises(RuntimeError):
        ncx.query.distance(ss, poses, ia, ib)

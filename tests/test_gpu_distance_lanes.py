"""Distances with one pair a lane (the scans of hulls shared by 8 lanes): batches around a wavefront
and above the partition's smallest, hulls of 4 to 256 vertices next to every other shape, with and
without a warm start under an iteration cap, against the oracle and the kernel with 8 lanes a pair."""
import numpy as np
import pytest
import torch

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from tests.test_gpu_parity import oracle_shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npairs,warm", [(1, False), (63, True), (65, False), (16384, True), (16384 + 63, False)])
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

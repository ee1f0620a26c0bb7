"""First hits of world rays where the traversal's scheduling has its edges: worlds of one and two
proxies, ray counts around a wavefront, a block and a refill, and a crowd in which every ray
reaches many capsules and hulls (more than a lane keeps, so that leaves go back onto its stack).
The oracle casts every shape whose stored box the ray enters and takes the least (toi, handle)."""
import numpy as np
import pytest
import torch

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from ncollide_amd.world import World
from tests.test_gpu_parity import oracle_shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nshapes,nrays,box", [(1, 1, 1.0), (1, 63, 1.0), (2, 65, 1.0), (3, 129, 1.0),
                                               (400, 1, 4.0), (400, 127, 2.0), (400, 3000, 2.0),
                                               (2000, 100003, 12.0)])
def test_world_first_rays_edges(ctx, orc, nshapes, nrays, box):
    w = workloads.full_pipeline(seed=50 + nshapes, n=nshapes, box=box, nclusters=1)
    ss = ncx.ShapeSet(records=w["records"], pool=w["pool"], ctx=ctx)
    world = World(ss, margin=0.05, prediction=0.0, max_pairs=1 << 18)
    p = w["poses"]
    poses = torch.as_tensor(p, device=ctx.device)
    world.step(poses)
    world.sync()
    stored = world.stored_aabbs().cpu().numpy().T.copy()
    rng = np.random.default_rng(nrays)
    tgt = p[rng.integers(0, nshapes, nrays), :3]
    ro = (tgt + rng.normal(0, 3, (nrays, 3))).astype(np.float32)
    ro[::5] = tgt[::5]  # from inside
    rd = ((tgt - ro) * rng.uniform(0.2, 1.5, (nrays, 1))).astype(np.float32)
    rd[::5] = rng.normal(size=(len(rd[::5]), 3)).astype(np.float32)
    oss = oracle_shapes(orc, w["records"], w["pool"])
    rh, rt, rn = orc.world_rays(oss, to_oracle_poses(p), stored, ro, rd, np.float32(20.0), 0)
    for o, d in ((ro, rd), (torch.as_tensor(ro, device=ctx.device), torch.as_tensor(rd, device=ctx.device))):
        h, t, n = world.first_interference_with_rays(poses, o, d, 20.0)
        assert np.array_equal(h.cpu().numpy().view(np.uint32), rh)
        assert np.array_equal(t.cpu().numpy().view(np.uint32), rt.view(np.uint32))
        assert np.array_equal(n.cpu().numpy().view(np.uint32), rn.view(np.uint32))


def _entries(boxes, o, d):
    """AABB::toi_with_ray (solid) of boxes the rays hit, in f32."""
    with np.errstate(divide="ignore", invalid="ignore"):
        inv = np.float32(1) / d
        a, b = (boxes[:, :3] - o) * inv, (boxes[:, 3:] - o) * inv
    return np.where(d != 0, np.minimum(a, b), 0).max(1).clip(min=0)


@pytest.mark.parametrize("size,away,early_hits", [(1.0, 3.0, 100), (0.05, 0.3, 30000), (8.0, 30.0, 0), (0.5, 100.0, 1000)])
def test_hits_before_their_boxes(ctx, orc, size, away, early_hits):
    """Casts that report a toi below their own box's entry (grazing capsules and hulls, small ones above
    all; balls from far away) in a crowd with tight boxes: the hit is the one with the least
    (max(toi, entry), toi, handle), whatever rays share a wavefront."""
    rng = np.random.default_rng(int(10 * size))
    n, nrays = 3000, 20000
    w = workloads.full_pipeline(seed=9, n=n, box=10.0, nclusters=1)
    rec, pool = w["records"], (w["pool"] * size).astype(np.float32)
    for k in ("p0", "p1", "p2"):
        rec[k] *= size
    t = rng.uniform(0, 6.0 * size, (n, 3))
    p = workloads.poses8(t, workloads.uniform_quats(rng, n)).astype(np.float32)
    ss = ncx.ShapeSet(records=rec, pool=pool, ctx=ctx)
    world = World(ss, margin=0.0, prediction=0.0, max_pairs=1 << 21)
    world.set_contacts(False)
    poses = torch.as_tensor(p, device=ctx.device)
    world.step(poses)
    world.sync()
    boxes = world.stored_aabbs().cpu().numpy().T.copy()
    ro = (3.0 * size + rng.normal(0, away, (nrays, 3))).astype(np.float32)
    rd = ((p[rng.integers(0, n, nrays), :3] + rng.normal(0, 0.3 * size, (nrays, 3)) - ro)
          * rng.uniform(0.2, 1.5, (nrays, 1))).astype(np.float32)
    oss = oracle_shapes(orc, rec, pool)
    cnt, h, toi, nrm = orc.world_rays(oss, to_oracle_poses(p), boxes, ro, rd, np.float32(20.0), 1)
    ray = np.repeat(np.arange(nrays), cnt)
    entry = _entries(boxes[h], ro[ray], rd[ray])
    order = np.lexsort((h, toi, np.maximum(toi, entry), ray))
    first = order[np.unique(ray[order], return_index=True)[1]]
    rh, rt, rn = np.full(nrays, 0xFFFFFFFF, np.uint32), np.full(nrays, -1, np.float32), np.zeros((nrays, 3), np.float32)
    rh[ray[first]], rt[ray[first]], rn[ray[first]] = h[first], toi[first], nrm[first]
    assert (toi < entry).sum() >= early_hits
    for k in (np.arange(nrays), rng.permutation(nrays)):  # the second time with other rays beside each
        gh, gt, gn = world.first_interference_with_rays(poses, ro[k], rd[k], 20.0)
        assert np.array_equal(gh.cpu().numpy().view(np.uint32), rh[k])
        assert np.array_equal(gt.cpu().numpy().view(np.uint32), rt[k].view(np.uint32))
        assert np.array_equal(gn.cpu().numpy().view(np.uint32), rn[k].view(np.uint32))
    # away from such hits the rule is the least (toi, handle) of all
    bh, bt, _ = orc.world_rays(oss, to_oracle_poses(p), boxes, ro, rd, np.float32(20.0), 0)
    assert size != 0.05 or (bt != rt).any()  # rays where the rule decides
    early = np.zeros(nrays, bool)
    early[ray[toi < entry]] = True
    assert np.array_equal(bh[~early], rh[~early]) and np.array_equal(bt[~early], rt[~early])


def test_world_without_shapes(ctx):
    ss = ncx.ShapeSet(records=np.zeros(0, ncx.shape.SHAPE_DTYPE), pool=np.zeros((0, 3), np.float32), ctx=ctx)
    world = World(ss, margin=0.0, prediction=0.0, max_pairs=1024)
    poses = torch.zeros((1, 8), device=ctx.device)
    world.step(poses)
    assert world.sync()[0] == 0
    o, d = np.zeros((70, 3), np.float32), np.ones((70, 3), np.float32)
    h, t, n = world.first_interference_with_rays(poses, o, d, 10.0)
    assert (h.cpu().numpy().view(np.uint32) == 0xFFFFFFFF).all() and (t == -1).all() and (n == 0).all()
    assert world.interferences_with_rays(poses, o, d, 10.0)[1].numel() == 0
    assert world.interferences_with_aabbs(np.array([[-9, -9, -9, 9, 9, 9]], np.float32))[1].numel() == 0

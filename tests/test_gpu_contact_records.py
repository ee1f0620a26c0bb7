"""Contacts in two kernels (GJK, then EPA on the records of the intersecting pairs): batches around
the wavefront and partition sizes, shape sets with pairs of some vertex-count buckets only, and the
EPA arenas' edges, against the oracle bit for bit."""
import numpy as np
import pytest

from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


def _scene(seed, types, n, nmax=64):
    from ncollide_amd import workloads
    from ncollide_amd.shape import CONVEX_HULL, SHAPE_DTYPE
    rng = np.random.default_rng(seed)
    pts, offs, cnts = workloads.ellipsoid_clouds(rng, 64, 8, nmax)
    pool, hoff, hcnt = workloads.build_hulls(pts, offs, cnts)
    rec = np.zeros(n, SHAPE_DTYPE)
    rec["type"] = rng.choice(types, n)
    p = rng.uniform(0.1, 0.6, (n, 3))
    rec["p0"], rec["p1"], rec["p2"] = p[:, 0], p[:, 1], p[:, 2]
    pick = rng.integers(0, 64, n)
    hull = rec["type"] == CONVEX_HULL
    rec["hull_offset"] = np.where(hull, hoff[pick], 0)
    rec["hull_count"] = np.where(hull, hcnt[pick], 0)
    t = rng.uniform(0, 0.8 * n ** (1 / 3), (n, 3))
    return rec, pool, workloads.poses8(t, workloads.uniform_quats(rng, n)), rng


def _check(ncx, rec, pool, poses, ia, ib, prediction=0.0, variant=None):
    import torch
    from ncollide_amd import query
    from ncollide_amd.math import to_oracle_poses
    ss = ncx.ShapeSet(records=rec, pool=pool)
    if variant is not None:
        ss.set_tuning([variant] * 4)
    g = query.contact(ss, torch.as_tensor(poses, device="cuda"), ia, ib, prediction)
    oss = orc.ShapeSet(rec["type"], np.stack([rec["p0"], rec["p1"], rec["p2"]], 1), rec["hull_offset"],
                       rec["hull_count"], pool, dtype=np.float32)
    r = orc.contact(oss, to_oracle_poses(poses), ia.astype(np.uint32), ib.astype(np.uint32), prediction)
    has = r["has"].astype(bool)
    assert np.array_equal(g["has_contact"].cpu().numpy(), has)
    gjk = (rec["type"][ia] != 0) & (rec["type"][ib] != 0)  # the oracle does not count a ball's projection
    assert np.array_equal(g["gjk_iters"].cpu().numpy()[gjk], r["gjk_iters"][gjk])
    for key in ("world1", "world2", "normal", "depth"):
        assert np.array_equal(g[key].cpu().numpy()[has], r[key][has]), key
        assert not g[key].cpu().numpy()[~has].any(), key
    return r


def _near_pairs(poses, n, npairs, rng):
    p = poses[:, :3].astype(np.float64)
    d = np.linalg.norm(p[:, None] - p[None], axis=2)
    d[np.tril_indices(n)] = np.inf
    k = np.argpartition(d, npairs, axis=None)[:npairs]
    ia, ib = np.divmod(k[rng.permutation(npairs)], n)
    return ia.astype(np.int32), ib.astype(np.int32)


@pytest.mark.parametrize("npairs", [1, 63, 64, 65, 1023, 4095, 4097, 16383, 16384, 16387])
def test_batch_sizes(npairs):
    import ncollide_amd as ncx
    n = max(16, npairs // 6)
    rec, pool, poses, rng = _scene(100 + npairs, [0, 1, 2, 3], n)
    ia, ib = _near_pairs(poses, n, npairs, rng)
    _check(ncx, rec, pool, poses, ia, ib)


@pytest.mark.parametrize("types,nmax", [([0, 1], 64), ([2], 64), ([3], 24), ([3], 250), ([0, 3], 250)])
def test_sets_with_some_buckets(types, nmax):
    import ncollide_amd as ncx
    rec, pool, poses, rng = _scene(7, types, 3000, nmax)
    ia, ib = _near_pairs(poses, 3000, 18000, rng)
    _check(ncx, rec, pool, poses, ia, ib, prediction=0.03)


@pytest.mark.parametrize("variant", range(5))
def test_runs_past_the_first_arena(variant):
    """Balls in capsules take 1 to a few hundred EPA iterations: runs that end in, and are saved
    by, each arena tier."""
    import ncollide_amd as ncx
    rec, pool, poses, rng = _scene(11, [0, 2], 4000)
    ia, ib = _near_pairs(poses, 4000, 20000, rng)
    r = _check(ncx, rec, pool, poses, ia, ib, variant=variant)
    it = r["epa_iters"]
    assert (it > 20).any() and (it > 40).any() and (it > 62).any() and ((it > 0) & (it < 20)).any()


@pytest.mark.parametrize("types,npairs", [([3], 20000), ([0, 1], 20000), ([3], 300)])
def test_bad_index_is_refused(types, npairs):
    """Whatever buckets the set's pairs fall in, and in batches that are partitioned or not."""
    import torch
    import ncollide_amd as ncx
    from ncollide_amd import query
    rec, pool, poses, rng = _scene(3, types, 200, 250)
    ss = ncx.ShapeSet(records=rec, pool=pool)
    p = torch.as_tensor(poses, device="cuda")
    ia, ib = rng.integers(0, 200, (2, npairs)).astype(np.int32)
    ib[npairs // 2] = 200
    v = torch.zeros((200, 3), device="cuda")
    for call in (lambda: query.contact(ss, p, ia, ib, 0.0), lambda: query.distance(ss, p, ia, ib),
                 lambda: query.time_of_impact(ss, p, v, ia, ib, 1.0)):
        with pytest.raises(ncx.NcxError):
            call()


@pytest.mark.parametrize("npairs", [1, 5000, 20000])
def test_set_without_shapes_refuses_pairs(npairs):
    import torch
    import ncollide_amd as ncx
    from ncollide_amd import query
    from ncollide_amd.shape import SHAPE_DTYPE
    ss = ncx.ShapeSet(records=np.zeros(0, SHAPE_DTYPE), pool=np.zeros((0, 3), np.float32))
    p = torch.zeros((1, 8), device="cuda")
    i = np.zeros(npairs, np.int32)
    for call in (lambda: query.contact(ss, p, i, i, 0.0), lambda: query.distance(ss, p, i, i),
                 lambda: query.time_of_impact(ss, p, torch.zeros((1, 3), device="cuda"), i, i, 1.0)):
        with pytest.raises(ncx.NcxError):
            call()

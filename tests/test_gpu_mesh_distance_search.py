"""The mesh distance search (k_md) where its bounds, lists and groups can go wrong: meshes of a few
triangles, query counts around a wavefront's groups, scattered triangles far from the origin, and
shapes near, far from and through the mesh, against the oracle bit for bit."""
import numpy as np
import pytest

import ncollide_amd as ncx
from ncollide_amd import workloads
from ncollide_amd.math import to_oracle_poses
from tests.test_gpu_parity import oracle_shapes

pytestmark = pytest.mark.gpu


def _check(ctx, orc, pts, tri, w, poses, idx, mpose):
    ss = ncx.ShapeSet(records=w["records"], pool=w["pool"], ctx=ctx)
    mesh = ncx.TriMesh(pts, tri, ctx=ctx)
    g = mesh.distance_to_shapes(ss, poses, idx, pose=mpose).cpu().numpy()
    oss = oracle_shapes(orc, w["records"], w["pool"])
    r = orc.mesh_distance(oss, pts, tri, to_oracle_poses(mpose.reshape(1, 8))[0], to_oracle_poses(poses), idx)
    assert np.array_equal(g.view(np.uint32), np.asarray(r, np.float32).view(np.uint32))
    return g


def _soup(rng, ntri, size, spread, centre):
    c = rng.uniform(-spread, spread, (ntri, 1, 3)) + np.asarray(centre)
    pts = (c + rng.normal(0, size, (ntri, 3, 3))).reshape(-1, 3).astype(np.float32)
    return pts, np.arange(3 * ntri, dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("ntri,n", [(1, 1), (1, 65), (2, 3), (3, 4), (5, 5), (40, 257), (700, 1000)])
@pytest.mark.parametrize("centre", [0.0, 300.0])
def test_scattered_triangles(ctx, orc, ntri, n, centre):
    rng = np.random.default_rng(1000 * ntri + n)
    pts, tri = _soup(rng, ntri, 0.6, 2.0, [centre, -centre, 0.5 * centre])
    w = workloads.full_pipeline(seed=ntri, n=max(n, 8), box=4.0, nclusters=1)
    poses = w["poses"].copy()
    # near and through the mesh, and some ten times farther
    far = np.where(np.arange(len(poses)) % 5 == 0, 10.0, 1.0)[:, None]
    poses[:, :3] = rng.uniform(-3.0, 3.0, (len(poses), 3)) * far + [centre, -centre, 0.5 * centre]
    mpose = np.zeros(8, np.float32)
    mpose[7] = 1.0
    idx = rng.integers(0, len(poses), n).astype(np.uint32)
    _check(ctx, orc, pts, tri, w, poses.astype(np.float32), idx, mpose)


@pytest.mark.parametrize("cells", [7, 60])
def test_shapes_around_a_terrain(ctx, orc, cells):
    rng = np.random.default_rng(cells)
    pts, tri = workloads.heightfield_mesh(seed=cells, cells=cells)
    w = workloads.full_pipeline(seed=cells, n=1500, box=4.0, nclusters=1)
    poses = w["poses"].copy()
    poses[:, :2] = rng.uniform(-0.1, 1.1, (1500, 2)) * 0.1 * cells
    poses[:, 2] = rng.uniform(-1.0, 4.0, 1500)
    ang = 0.4
    mpose = np.array([0.5, 0.2, -0.3, 0.0, np.sin(ang / 2), 0.0, 0.0, np.cos(ang / 2)], np.float32)
    g = _check(ctx, orc, pts, tri, w, poses.astype(np.float32), np.arange(1500, dtype=np.uint32), mpose)
    assert (g > 0.5).any() and ((g > 0) & (g < 0.2)).any() and (g == 0).any()


@pytest.mark.parametrize("mesh,n", [("floor", 600000), ("sheets", 20000)])
def test_shapes_near_large_triangles(ctx, orc, mesh, n):
    """GJK in f32 reports a zero distance for some shapes that are apart from a triangle much larger
    than they are, also where another triangle is nearer.  Whether such a triangle decides is the
    reference's order of search (least cost first), not the order in which lanes come to them."""
    rng = np.random.default_rng(1)
    if mesh == "floor":  # eight triangles
        X, Y = np.meshgrid(np.arange(3) * 100.0, np.arange(3) * 100.0)
        pts = np.stack([X.ravel(), Y.ravel(), rng.uniform(-5, 5, 9)], 1).astype(np.float32)
        p = np.array([0, 1, 3, 4])
        tri = np.concatenate([np.stack([p, p + 1, p + 3], 1), np.stack([p + 1, p + 4, p + 3], 1)]).astype(np.uint32)
        bary = rng.dirichlet([1, 1, 1], n)[:, :, None]
        t = (pts[tri[rng.integers(0, 8, n)]] * bary).sum(1)
        t[:, 2] += rng.uniform(-2, 2, n)
    else:  # 256 nearly parallel ones within 0.2 of each other, the shapes on one side
        T = rng.normal(0, 100.0, (256, 3, 3))
        T[:, :, 2] = rng.uniform(-0.2, 0, (256, 1)) + rng.normal(0, 0.02, (256, 3))
        t = np.concatenate([rng.normal(0, 30.0, (n, 2)), rng.uniform(0.1, 0.8, (n, 1))], 1)
        rot = np.linalg.qr(rng.normal(size=(3, 3)))[0]
        t = t @ rot.T
        pts = (T.reshape(-1, 3) @ rot.T).astype(np.float32)
        tri = np.arange(768, dtype=np.uint32).reshape(-1, 3)
    w = workloads.full_pipeline(seed=3, n=20000, box=60.0, nclusters=4)
    w = {"records": np.tile(w["records"], n // 20000), "pool": w["pool"]}
    poses = workloads.poses8(t, workloads.uniform_quats(rng, n)).astype(np.float32)
    mpose = np.zeros(8, np.float32)
    mpose[7] = 1.0
    idx = np.arange(n, dtype=np.uint32)
    g = _check(ctx, orc, pts, tri, w, poses, idx, mpose)
    exact = orc.mesh_distance(oracle_shapes(orc, w["records"], w["pool"], np.float64), pts.astype(np.float64), tri,
                              to_oracle_poses(mpose.reshape(1, 8))[0].astype(np.float64),
                              to_oracle_poses(poses).astype(np.float64), idx)
    assert (g[exact > 1e-4] == 0).any()  # such zeros are among the queries
    order = rng.permutation(n)  # other queries beside each
    again = _check(ctx, orc, pts, tri, w, poses, order.astype(np.uint32), mpose)
    assert np.array_equal(again.view(np.uint32), g[order].view(np.uint32))
